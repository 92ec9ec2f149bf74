"""The 32-bit products on the matrix cores (streaming kernel up to 64 rows, tiles beyond) against the kernel of the vector
ALU's FMAs, which weights that do not start at 16 bytes still run through: the same bits."""
import pytest
import torch

from hector_engine_amd.kernels import ops

pytestmark = pytest.mark.gpu


def operands(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    a, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    a[::3] *= 1e-20                     # rows whose products are denormal, rows of large ones, zeros of both signs
    w[::4] *= 1e-20
    a[1::5] *= 1e15
    a[:, ::7] = 0.0
    w[:, ::5] = -0.0
    return a.cuda(), w.cuda(), torch.randn(N, generator=g).cuda()


def by_fma(a, w, bias):
    """The product through the FMA kernel, eight rows at a time."""
    N, K = w.shape
    shifted = torch.empty(N * K + 1, device="cuda")[1:].view(N, K)
    shifted.copy_(w)
    assert shifted.data_ptr() % 16 != 0
    out = torch.empty(a.shape[0], N, device="cuda")
    for r in range(0, a.shape[0], 8):
        m = min(8, a.shape[0] - r)
        ops.gemm_plain(out[r:r + m], a[r:r + m], shifted, bias, m,
                       workspace=torch.empty(ops.gemm_plain_workspace_floats(m, N, K), device="cuda"))
    return out


@pytest.mark.parametrize("M", [1, 2, 9, 16, 17, 32, 33, 63, 64, 65, 127, 128, 129, 300])
@pytest.mark.parametrize("N,K", [(16, 128), (5, 256), (100, 1152), (4110, 384), (129, 2048 + 128)])
def test_the_matrix_cores_give_the_bits_of_the_fma_chain(M, N, K):
    a, w, bias = operands(M, N, K, M * N + K)
    want = by_fma(a, w, bias)
    out = torch.full((M, N), 7.0, device="cuda")
    ops.gemm_plain(out, a, w, bias, M)
    assert torch.equal(out.view(torch.int32), want.view(torch.int32))
    ops.gemm_plain(out, a, w, None, M)
    assert torch.equal(out.view(torch.int32), by_fma(a, w, None).view(torch.int32))


@pytest.mark.parametrize("M", [9, 64, 65, 130])
@pytest.mark.parametrize("N,K", [(33, 31), (130, 100), (65, 129), (64, 260)])
def test_widths_that_are_no_multiple_of_a_stage_run_in_tiles(M, N, K):
    a, w, bias = operands(M, N, K, M + N + K)
    out = torch.full((M, N), 7.0, device="cuda")
    ops.gemm_plain(out, a, w, bias, M)
    assert torch.equal(out.view(torch.int32), by_fma(a, w, bias).view(torch.int32))


def test_what_is_not_finite_stays_in_its_row_and_column():
    a, w, _ = operands(70, 40, 256, 1)
    a[3, 5], a[9, 200], w[7, 0] = float("inf"), float("nan"), float("-inf")
    want = by_fma(a, w, None)
    for M in (20, 70):
        out = torch.empty(M, 40, device="cuda")
        ops.gemm_plain(out, a[:M], w, None, M)
        assert torch.equal(out.isnan(), want[:M].isnan()) and torch.equal(out.nan_to_num(1.0, 2.0, 3.0), want[:M].nan_to_num(1.0, 2.0, 3.0))


@pytest.mark.parametrize("M", [1, 3, 4, 8, 9, 33, 64])
@pytest.mark.parametrize("N,K", [(24580, 128), (24576, 256), (16400, 512), (300, 3072), (1500, 4096)])
def test_few_segments_and_few_weight_rows_give_the_same_bits_with_and_without_a_workspace(M, N, K):
    a, w, bias = operands(M, N, K, M + N + K)
    want = by_fma(a, w, bias)
    out = torch.full((M, N), 7.0, device="cuda")
    floats = ops.gemm_plain_workspace_floats(M, N, K, a=a, w=w, out=out)
    for workspace in ({None, floats} if floats else {None}):
        out.fill_(7.0)
        ops.gemm_plain(out, a, w, bias, M, workspace=workspace and torch.full((workspace,), float("nan"), device="cuda"))
        assert torch.equal(out.view(torch.int32), want.view(torch.int32))
