"""float32 x by bfloat16 w as three products of bfloat16 numbers (``csrc/gemm_split.hip``): edges of tiles, blocks and chunks, the same bits
for every number of rows, errors no larger than the float32 instruction's, and entries that have no three parts."""
import pytest
import torch

from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def product(x, w):
    return ops.gemm(x, w, torch.float32)


@pytest.mark.parametrize("M", [1, 15, 16, 17, 63, 65, 200])
@pytest.mark.parametrize("N,K", [(1, 32), (63, 224), (129, 256), (300, 288), (1000, 1024), (40000, 96)])
def test_edges(M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    x = (torch.randn(M, K, generator=g) * torch.exp(3 * torch.randn(M, K, generator=g))).to(DEV)
    w = torch.randn(N, K, generator=g).bfloat16().to(DEV)
    got, want = product(x, w), x.double() @ w.double().T
    # K products, exact, added in float32: each addition is off by 2^-24 of a sum that is no larger than the terms' absolute values
    allowed = 2.0 ** -24 * K * (x.double().abs() @ w.double().abs().T)
    assert bool(((got.double() - want).abs() <= allowed).all())
    plain = product(x, w.float())           # float32 by float32, on the float32 instruction
    if M * N >= 10000:      # a root mean square over n errors is itself off by some 1 / sqrt(2 n) of it: 0.7 % here, 20 % at 15 entries
        assert float((got.double() - want).norm()) <= 1.05 * float((plain.double() - want).norm())
    # a row alone, few rows and many have the same bits
    many = product(x.repeat(-(-700 // M), 1), w)
    assert torch.equal(many[:M], got) and torch.equal(many[-M:], got)
    assert torch.equal(product(x[M // 2:M // 2 + 1].contiguous(), w)[0], got[M // 2])


@pytest.mark.parametrize("M", [7, 40])
@pytest.mark.parametrize("K", [288, 4096])
def test_entries_without_parts(M, K):
    """Infinite and not-a-number entries reach the outputs that 64 bits give them to; the largest and the smallest numbers, each with rows of
    their own that hold nothing larger, lose nothing."""
    g = torch.Generator().manual_seed(K)
    x, w = torch.randn(M, K, generator=g).to(DEV), torch.randn(130, K, generator=g).bfloat16().to(DEV)
    x[0, 5], x[1, 270], x[2, 7] = float("inf"), float("nan"), -float("inf")
    w[3, 9], w[4, 271] = float("inf"), float("nan")
    w[5, 5] = 0.0
    x[3, 20:22] = torch.tensor([3.4028235e38, -3.4028235e38])
    w[:, 20] = 2.0 ** -10
    w[:, 21] = 2.0 ** -12
    x[4] *= 1e-36
    x[5] *= 1.2e-38
    x[6] *= 1e-41
    got, want = product(x, w).double(), x.double() @ w.double().T
    same = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isposinf(got), torch.isposinf(want))
    assert torch.equal(torch.isneginf(got), torch.isneginf(want))
    assert bool(same[3:].any(dim=1).all()), "every row has outputs to compare"
    # as in test_edges, and the results, chunk by chunk, rounded to multiples of 2^-149
    allowed = 2.0 ** -24 * K * (x.double().abs() @ w.double().abs().T) + 2.0 ** -149 * (1 + K // 256)
    assert bool(((got - want).abs()[same] <= allowed[same]).all())
