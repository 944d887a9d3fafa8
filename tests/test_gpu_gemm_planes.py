"""float32 x by bfloat16 w where x's three parts are cut beforehand, and by eight waves: the bits of the kernel for few rows, edges of
tiles, chunks that are not whole, and numbers that have no three parts."""
import pytest
import torch

from lucciola_amd.kernels import ops

pytestmark = pytest.mark.gpu


def _operands(M, N, K, offset=0):
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M * K + offset, device="cuda", generator=gen)[offset:].view(M, K)
    return x, (torch.randn(N, K, device="cuda", generator=gen) * 0.05).to(torch.bfloat16)


@pytest.mark.parametrize("M,N,K,offset", [(200, 50001, 96, 0), (193, 49920, 352, 0), (250, 70001, 64, 0), (256, 60000, 1024, 0),
                                          (200, 50001, 96, 1)])
def test_planes(M, N, K, offset):
    x, w = _operands(M, N, K, offset)
    assert ops.library().lc_gemm_generic_workspace(M, N, K) == (3 * M * K + 1) // 2       # by planes
    got = ops.gemm(x, w, torch.float32)
    for first in (0, 64, 128, M - 9):       # up to 16 rows have a kernel of their own, with the same additions
        few = x[first:first + 9].clone()
        assert torch.equal(got[first:first + 9], ops.gemm(few, w, torch.float32))
    want = x[:, None, :].double() @ w[::997].double().T[None]       # a column of every tile and more
    sizes = x.double().abs() @ w[::997].double().abs().T
    assert bool(((got[:, ::997].double() - want[:, 0]).abs() <= sizes * K * 2.0 ** -24).all())


@pytest.mark.parametrize("M,N,K", [(200, 50001, 352), (566, 3000, 96)])
def test_numbers_without_three_parts(M, N, K):
    x, w = _operands(M, N, K)
    x[5, 7], x[70, 40], x[M - 1, 95], x[M - 2, 3] = float("inf"), float("nan"), 3e38, 1e-41
    got = ops.gemm(x, w, torch.float32)
    for row in (5, 70, M - 1, M - 2, 0, 69, 71):
        assert torch.equal(got[row].nan_to_num(nan=12345.0), ops.gemm(x[row:row + 1].clone(), w, torch.float32)[0].nan_to_num(nan=12345.0))
    assert bool(got[70].isnan().all()) and bool(got[0].isfinite().all())


@pytest.mark.parametrize("M,N,K", [(65, 8200, 96), (566, 6144, 256), (130, 1025, 2048), (64, 20000, 64), (17, 6144, 1024)])
def test_eight_waves(M, N, K):
    """More than a workgroup a CU in tiles of 64 x 64: tiles of 64 x 128, whole and with their chunks shared out."""
    x, w = _operands(M, N, K)
    got = ops.gemm(x, w, torch.float32)
    for first in (0, M - 11):
        assert torch.equal(got[first:first + 11], ops.gemm(x[first:first + 11].clone(), w, torch.float32))
    want, sizes = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert bool(((got.double() - want).abs() <= sizes * K * 2.0 ** -24).all())


def test_planes_stay_in_registers():
    """The kernel's operands land in registers behind the compiler's back: with scratch memory the products go by tiles."""
    assert ops.library().lc_gemm_planes_ok() == 1


def test_room_for_planes():
    """Only the types that are multiplied by planes ask for room, and never for more than 256 MiB: more rows go one portion after the other, with
    the same bits."""
    lib, f32, bf16 = ops.library(), ops.DT_F32, ops.DT_BF16
    M, N, K = 512, 65000, 1024
    assert lib.lc_gemm_generic_workspace_of(M, f32, N, bf16, K, f32) == (3 * M * K + 1) // 2
    for types in ((f32, f32, f32), (bf16, f32, f32), (bf16, f32, bf16), (bf16, bf16, f32), (bf16, bf16, bf16)):
        assert lib.lc_gemm_generic_workspace_of(M, types[0], N, types[1], K, types[2]) == 0
    M, N, K = 1500, 5000, 32768
    assert (3 * M * K + 1) // 2 > 1 << 26 >= lib.lc_gemm_generic_workspace_of(M, f32, N, bf16, K, f32) > 0
    x, w = _operands(M, N, K)
    got = ops.gemm(x, w, torch.float32)
    for first in (0, 1270, 1355, 1365, M - 9):
        assert torch.equal(got[first:first + 9], ops.gemm(x[first:first + 9].clone(), w, torch.float32))
