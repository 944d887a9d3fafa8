"""Masked attention on the matrix cores (``csrc/masked_attention_bf16.hip``) at the lines of its dispatch: few and many heads a kv head, for which
a wave takes one block of keys a step or two, and steps of lone tokens that are all on the card at once or are not."""
import pytest
import torch

from lucciola_amd.engine.batch import HostLayout, Plan
from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def both(history, fresh, heads, kv, maps, d, dv, window=0):
    """The matrix cores' result and the general kernel's, and the values' largest entry."""
    page, R = 16, len(fresh)
    pages = [-(-(h + f) // page) for h, f in zip(history, fresh)]
    table, at = torch.zeros((R, max(pages)), dtype=torch.int32), 0
    for r, n in enumerate(pages):
        table[r, :n] = torch.arange(at, at + n)
        at += n
    g = torch.Generator(device=DEV).manual_seed(heads + kv + d + dv + R)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    kc, vc = rand(at, page, kv * maps * d), rand(at, kv * dv, page)
    q_start = [0]
    for f in fresh:
        q_start.append(q_start[-1] + f)
    tok = torch.tensor([r for r, f in enumerate(fresh) for _ in range(f)], dtype=torch.int32, device=DEV)
    pos = torch.tensor([history[r] + i for r, f in enumerate(fresh) for i in range(f)], dtype=torch.int32, device=DEV)
    q = rand(q_start[-1], heads * maps * d)
    arrays, info = ops.plan_latent_attention(HostLayout(R, q_start[-1], q_start, history, page, False))
    plan = Plan({k: torch.from_numpy(v).to(DEV) for k, v in arrays.items()}, info)
    longest = max(h + f for h, f in zip(history, fresh))
    call = lambda: ops.masked_attention(q, kc, vc, tok, pos, table.to(DEV), page, heads, kv, maps, d, dv, d ** -0.5, window=window,
                                        subtract=0.3 if maps == 2 else 0.0, plan=plan, max_ctx=longest)
    fast = call()
    before = ops.masked_attention_matrix_cores(False)
    try:
        return fast, call(), float(vc.abs().max())
    finally:
        ops.masked_attention_matrix_cores(before)


def near(fast, plain, largest):
    # both are rounded to bfloat16 (half a unit each, 2^-8 of the entry), and the weights of the one are good to 2^-15; sums cancel
    allowed = 2.0 ** -7 * plain.float().abs() + 2.0 ** -12 * largest
    assert float(((fast.float() - plain.float()).abs() / allowed).max()) <= 1.0


@pytest.mark.parametrize("heads,kv", [(3, 3), (4, 2), (3, 1), (4, 1), (16, 2), (5, 1)])
@pytest.mark.parametrize("maps,d,dv", [(1, 64, 64), (1, 64, 32), (1, 128, 32), (2, 128, 64), (2, 64, 32), (1, 128, 128), (2, 64, 128)])
def test_heads_a_kv_head(heads, kv, maps, d, dv):
    near(*both([0, 70, 300, 9], [100, 33, 17, 1], heads, kv, maps, d, dv))


@pytest.mark.parametrize("requests,kv", [(1, 3), (7, 4), (9, 4), (64, 4), (65, 4), (128, 4), (129, 4), (200, 16), (1030, 1)])
@pytest.mark.parametrize("window", [0, 100])
def test_lone_tokens(requests, kv, window):
    history = [1 + (37 * r) % 700 for r in range(requests)]
    near(*both(history, [1] * requests, 2 * kv, kv, 1, 64, 32, window))
