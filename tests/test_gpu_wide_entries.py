"""Element-wise kernels with several entries a thread: sizes that are and are not whole pieces, and rows that are not aligned."""
import pytest
import torch

from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


def near(got, want, dtype, atol=1e-6):
    # half a unit of bfloat16 where results are rounded; float32: some ten roundings on the way
    torch.testing.assert_close(got.double(), want, rtol=2.0 ** -8 if dtype == torch.bfloat16 else 2e-6, atol=atol)


def gelu(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,I", [(1, 8), (3, 24), (5, 25), (70, 2048), (300, 2056), (2, 4100), (9001, 64), (33000, 24), (4000, 136)])
def test_gated(dtype, T, I):
    g = torch.Generator().manual_seed(T + I)
    gu = (torch.randn(T, 2 * I, generator=g) * 4).to(dtype).to(DEV)
    for rows in (gu, torch.empty(T * 2 * I + 1, dtype=dtype, device=DEV)[1:].view(T, 2 * I).copy_(gu)):      # the second is not aligned
        gate, up = gu.double()[:, :I], gu.double()[:, I:]
        near(ops.gated_activation(rows, "silu"), torch.nn.functional.silu(gate) * up, dtype)
        # in float32 1 + tanh is off by 2^-24 however small it is, and is taken times half of gate and up
        near(ops.gated_activation(rows, "gelu_tanh"), gelu(gate) * up, dtype, 1e-6 + 2.0 ** -24 * float(gate.abs().max() * up.abs().max()))
        held, shifted = gate.clamp(max=3.0), up.clamp(-3.0, 3.0) + 1.0
        near(ops.gated_activation(rows, "silu", ops.GateForm(3.0, 1.7, 1.0)), held * torch.sigmoid(1.7 * held) * shifted, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [1, 8, 31, 4096, 100003, 1 << 20, (1 << 20) + 8, (1 << 20) + 9])
def test_activation(dtype, n):
    x = (torch.randn(1, n, generator=torch.Generator().manual_seed(n)) * 4).to(dtype).to(DEV)
    for kind, f in ((1, gelu), (2, lambda z: torch.relu(z) ** 2), (6, torch.nn.functional.gelu)):
        y = x.clone()
        ops._call("lc_activation", ops._ptr(y), ops._dt(y), kind, 0.0, 0.0, y.numel(), ops._stream())
        near(y, f(x.double()), dtype, 1e-6 + 2.0 ** -24 * float(x.abs().max()))       # 1 + tanh, 1 + erf: as above


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,top,n", [(1, 1, 4), (7, 3, 66), (40, 4, 2048), (5, 2, 4100), (9, 2, 301), (6, 8, 2050), (3, 7, 512)])
def test_combine(dtype, T, top, n):
    g = torch.Generator().manual_seed(T + n)
    E = top + 2
    routing = ops.moe_route(torch.randn(T, E, generator=g).to(DEV), top, True)
    y = torch.randn(T * top, n, generator=g).to(DEV)
    shared, gates = torch.randn(T, n, generator=g).to(dtype).to(DEV), torch.randn(T, 3, generator=g).to(DEV)
    rows = y.double()[routing.entry_row.long()].view(T, top, n)
    weighed = (rows * routing.weights.double()[:, :, None]).sum(1)
    near(ops.moe_combine(y, routing, dtype), weighed, dtype)
    got = ops.moe_combine_shared(y, routing, shared, gates, 2, dtype, weighted=True)
    near(got, weighed + torch.sigmoid(gates.double()[:, 2:]) * shared.double(), dtype)
    near(ops.moe_combine_shared(y, routing, None, None, 0, dtype, weighted=False), rows.sum(1), dtype)
