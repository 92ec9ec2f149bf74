"""bf16 products of some hundred rows and few columns in tiles that are one round of the chip."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from hector_engine_amd.kernels import ops
    return ops


def product(ops, M, N, K, bias, tile, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M + 3, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    b = None if bias is None else torch.randn(N, generator=g, device="cuda").to(bias)
    out = torch.full((M + 2, N), 77.0, dtype=torch.bfloat16, device="cuda")
    ops.gemm_few_tiles(out, x, w, b, M, tile)
    want = x[:M].double() @ w.double().t() + (0 if b is None else b.double())
    # a bf16 result of fp32 sums: half an ulp (2^-9) of the result and K 2^-24 of the sum of the products' sizes (some 1 here)
    assert torch.allclose(out[:M].double(), want, rtol=2 ** -8, atol=2 ** -14)
    assert bool((out[M:] == 77).all())


@pytest.mark.parametrize("bm", [64, 128])
@pytest.mark.parametrize("bn", [32, 48, 64, 80, 96, 112, 128])
@pytest.mark.parametrize("K,bias", [(64, None), (192, torch.bfloat16), (576, torch.float32)])
def test_every_tile_at_its_edges(ops, bm, bn, K, bias):
    """Whole tiles, one row and four columns more, and less than one tile; fewer stages of K than are in flight, and more."""
    for M, N in ((bm, bn), (2 * bm + 1, 3 * bn + 4), (bm - 1, bn - 4), (1, 4)):
        product(ops, M, N, K, bias, bm << 16 | bn, seed=M + N)


@pytest.mark.parametrize("M,N,K", [(65, 896, 896), (256, 4608, 3584), (512, 1152, 896), (300, 5120, 1024), (1000, 896, 4864)])
def test_chosen_tiles(ops, M, N, K):
    tile = ops.few_tiles_tile(M, N)
    bm, bn = tile >> 16, tile & 0xffff
    assert tile and -(-M // bm) * -(-N // bn) <= ops.compute_units()
    product(ops, M, N, K, torch.bfloat16, tile)


def test_what_the_rule_takes(ops):
    """One round of tiles, from half of the chip's units on where K is long; nothing that cannot be read where it lies."""
    from hector_engine_amd.parts.linear import Linear
    bf16 = torch.bfloat16

    def tile(M, N, K, out_dtype=bf16, at=0):
        x = torch.empty(M * K + 8, dtype=bf16, device="cuda")[at:at + M * K].view(M, K)
        return Linear(torch.empty(N, K, dtype=bf16, device="cuda"))._few_tiles(M, x, torch.empty(M, N, dtype=out_dtype, device="cuda"), out_dtype)

    assert tile(256, 4608, 3584) == 64 << 16 | 80 and tile(128, 3584, 3584) == 64 << 16 | 32
    assert tile(100, 64, 1024) and not tile(100, 64, 1088)           # four tiles
    assert not tile(256, 4608, 5184) and not tile(256, 4608, 3584 + 32)
    assert not tile(256, 4610, 3584) and not tile(256, 4608, 3584, torch.float32)
    assert not tile(256, 4608, 3584, at=1)                           # off 16-byte boundaries
    assert not tile(2048, 4608, 3584) and not tile(256, 37888, 3584)  # more than a round


def test_refusals(ops):
    from hector_engine_amd.kernels.lib import KernelLibraryError
    x, w, out = (torch.empty(64, n, dtype=torch.bfloat16, device="cuda") for n in (128, 128, 64))
    with pytest.raises(KernelLibraryError, match="no tiles"):
        ops.gemm_few_tiles(out, x, w, None, 64, 64 << 16 | 40)
    with pytest.raises(KernelLibraryError, match="bad sizes"):
        ops.gemm_few_tiles(out[:, :63].contiguous(), x, w[:63].contiguous(), None, 64, 64 << 16 | 64)
