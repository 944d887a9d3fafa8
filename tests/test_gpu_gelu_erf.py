"""The exact GELU of bfloat16 results, written without erf, over its whole range, and no less exact in float32 than with
the library's erf."""
import pytest
import torch

from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu


def test_gelu_for_bfloat16():
    """Half a unit of bfloat16 (2^-9) and what float32 leaves below -1 (7e-6, see the kernel): one unit at ties.  Results below the
    smallest normal number may be zero."""
    z = torch.cat([torch.linspace(-14, 14, 400001), torch.logspace(-30, 4, 5001), -torch.logspace(-30, 4, 5001),
                   torch.tensor([0.0, -0.0, 1e30, -1e30])]).to(torch.bfloat16)
    got = z.cuda()
    ops.activation(got, "gelu")
    x = z.double()
    want = x * 0.5 * torch.special.erfc(-x * 0.5 ** 0.5)
    assert bool(((got.cpu().double() - want).abs() <= want.abs() * (2.0 ** -8 + 1e-5) + 2.0 ** -125).all())
    special = torch.tensor([float("inf"), float("nan")], dtype=torch.bfloat16, device="cuda")
    ops.activation(special, "gelu")
    assert float(special[0]) == float("inf") and bool(special[1].isnan())


def test_gelu_is_as_exact_as_with_erf():
    """Float32 arguments in (-1, 1), which an experts' product makes exactly out of bfloat16 parts: a result is rounded to the wrong neighbour
    where the correct one lies within the formula's error of a boundary, and boundaries are 2^-8 to 2^-7 of the result apart (185 to a
    result in the mean).  A mean error of 0.6e-7 (erff: 0.4e-7; with an unrefined 1 / (1 + c |z|) to the power of up to nine: 1.0e-7) makes
    0.6e-7 * 185 of the results wrong."""
    T, N, K = 512, 8192, 64
    gen = torch.Generator().manual_seed(3)
    high = torch.arange(-256, 256).double() / 256
    low = torch.randint(0, 256, (2, N), generator=gen).double() * torch.tensor([[2.0 ** -16], [2.0 ** -23]])
    x, w = torch.zeros(T, K), torch.zeros(1, N, K)
    x[:, 0], x[:, 1], x[:, 2], w[0, :, 0] = high.float(), 1, 1, 1
    w[0, :, 1:3] = low.t().float()
    routing = ops.moe_route(torch.zeros(T, 1, device="cuda"), 1, large_tiles=True)
    got = ops.moe_experts(x.bfloat16().cuda(), w.bfloat16().cuda(), routing, torch.bfloat16, activation="gelu", gather=True)
    rows = torch.empty(T, N, dtype=torch.bfloat16, device="cuda")
    rows[routing.sorted_token.long()] = got
    z = (high[:, None] + low.sum(0)[None]).cuda()
    assert torch.equal(z, z.float().double())
    want = (z * 0.5 * torch.special.erfc(-z * 0.5 ** 0.5)).bfloat16()
    assert int((rows != want).sum()) <= 0.6e-7 * 185 * T * N
