"""Layer norms and dynamic tanh over rows in 16-byte pieces and entry by entry, against float64."""
import pytest
import torch

from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _rows(T, n, offset, dtype, gen):
    """[T, n] that begins `offset` entries behind an aligned place."""
    return torch.randn(T * n + offset, device="cuda", generator=gen)[offset:].to(dtype).view(T, n) if not offset else \
        torch.randn(T * n + offset, device="cuda", generator=gen).to(dtype)[offset:].view(T, n)


@pytest.mark.parametrize("n,offset", [(8, 0), (2048, 0), (2040, 0), (4096, 0), (8192, 0), (2047, 0), (2048, 1), (9000, 0), (64, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("normed", [True, False])
def test_layer_norm(n, offset, dtype, normed):
    gen = torch.Generator(device="cuda").manual_seed(n + offset)
    T = 5
    h, d = _rows(T, n, offset, torch.float32, gen), _rows(T, n, offset, dtype, gen)
    w, b, pw, pb = (torch.randn(n, device="cuda", generator=gen) for _ in range(4))
    want_h = h.double()
    delta = d.double()
    if normed:
        delta = torch.nn.functional.layer_norm(delta, (n,), pw.double(), pb.double(), 1e-5)
    want_h = want_h + delta
    want = torch.nn.functional.layer_norm(want_h, (n,), w.double(), b.double(), 1e-5)
    got = ops.layer_norm(h, ops.NormedBranch(d, pw, pb, 1e-5) if normed else d, w, b, 1e-5, dtype)
    # sums of n numbers of size one in float32: 2^-24 sqrt(n) of the deviation, some ten roundings beside; then the result's own type
    close = 1e-5 * (1 + w.abs().double() * 4)
    assert bool(((h.double() - want_h).abs() <= 1e-5 * (1 + want_h.abs())).all())
    assert bool(((got.double() - want).abs() <= close + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else want.abs() * 1e-5)).all())


@pytest.mark.parametrize("T,n,offset", [(300, 8, 0), (300, 2048, 0), (257, 2044, 0), (300, 2047, 0), (300, 64, 1), (3, 2048, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_dynamic_tanh(T, n, offset, dtype):
    gen = torch.Generator(device="cuda").manual_seed(T + n)
    h, d = _rows(T, n, offset, torch.float32, gen) * 2, _rows(T, n, offset, dtype, gen)
    h[0, :4] = torch.tensor([1e-6, -1e-4, 30.0, -30.0])
    d[0, :4] = 0
    w, b = torch.randn(n, device="cuda", generator=gen), torch.zeros(n, device="cuda")
    want_h = h.double() + d.double()
    got = ops.dynamic_tanh(h, d, w, b, 0.5, dtype)
    assert bool(((h.double() - want_h).abs() <= 2.0 ** -24 * want_h.abs()).all())
    want = torch.tanh(0.5 * want_h) * w.double()
    assert bool(((got.double() - want).abs() <= want.abs() * (2.0 ** -8 + 2e-6 if dtype == torch.bfloat16 else 1e-6) + 1e-30).all())


@pytest.mark.parametrize("T", [3, 300])
def test_dynamic_tanh_of_bfloat16_rounds_what_float32_gives(T):
    """The tanh of bfloat16 results is the one of float32 results: nothing of it is less exact."""
    gen = torch.Generator(device="cuda").manual_seed(T)
    n = 2048
    h = torch.randn(T, n, device="cuda", generator=gen) * 2
    w, b = torch.ones(n, device="cuda"), torch.zeros(n, device="cuda")
    exact = ops.dynamic_tanh(h.clone(), None, w, b, 0.5, torch.float32)
    assert torch.equal(ops.dynamic_tanh(h.clone(), None, w, b, 0.5, torch.bfloat16), exact.to(torch.bfloat16))
