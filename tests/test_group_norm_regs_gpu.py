"""Norms by groups, gated sums and polynomial norms whose elements are held in registers: every count of elements a lane holds."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64


def gn(x, groups, eps):
    parts = x.reshape(len(x), groups, -1)
    return (parts / torch.sqrt((parts * parts).mean(-1, keepdim=True) + eps)).reshape(x.shape)


def close(got, want, dtype):
    # fp32 sums of up to 4096 squares (a butterfly over chains of up to 64: some 1e-6), a result rounded to bf16 (half an ulp, 2^-9)
    tol = 2 ** -8 if dtype == BF16 else 4e-6
    assert torch.allclose(got.cpu().to(F64), want, rtol=tol, atol=tol)


@pytest.mark.parametrize("width", [1, 63, 64, 65, 128, 129, 257, 512, 513, 1024, 1025, 2048, 2049])
@pytest.mark.parametrize("rows,groups,next_groups", [(3, 3, 3), (70, 2, 2), (3, 2, 1), (70, 5, 5)])
def test_add_group_normed(width, rows, groups, next_groups):
    from hector_engine_amd.kernels import ops
    D = width * groups
    g = torch.Generator().manual_seed(D)
    resid, weight, follow = torch.randn(rows, D, generator=g), torch.randn(D, generator=g), torch.randn(D, generator=g)
    for dt, ot, norm in ((BF16, F32, False), (BF16, BF16, True), (F32, BF16, True), (None, BF16, True), (F32, None, False)):
        delta = None if dt is None else torch.randn(rows, D, generator=g).to(dt)
        r, out = resid.cuda(), None if ot is None else torch.full((rows, D), 7.0, dtype=ot, device="cuda")
        ops.add_group_normed(r, None if delta is None else delta.cuda(), None if delta is None else weight.cuda(), groups, 1e-3, 0.5, out, rows,
                             next_weight=follow.cuda() if norm else None, next_groups=next_groups, next_eps=1e-2)
        want = resid.to(F64)
        if delta is not None:
            want = want + 0.5 * gn(delta.to(F64), groups, 1e-3) * weight.to(F64)
        close(r, want, F32)
        if out is not None:
            close(out, gn(want, next_groups, 1e-2) * follow.to(F64) if norm else want, ot)


@pytest.mark.parametrize("width,groups", [(1025, 1), (1537, 2), (2048, 1), (2048, 4)])
@pytest.mark.parametrize("dt,ot", [(BF16, BF16), (F32, F32), (None, BF16)])
def test_rows_have_the_same_bits_in_any_company(width, groups, dt, ot):
    """More than 16 elements a lane are held in registers up to 64 rows and read again beyond: the same rows in a step of 64 and in one of 130."""
    from hector_engine_amd.kernels import ops
    D = width * groups
    g = torch.Generator().manual_seed(D)
    resid, weight, follow = torch.randn(130, D, generator=g), torch.randn(D, generator=g).cuda(), torch.randn(D, generator=g).cuda()
    delta = None if dt is None else torch.randn(130, D, generator=g).to(dt)
    got = {}
    for rows in (64, 130):
        r, out = resid[:rows].cuda(), torch.empty(rows, D, dtype=ot, device="cuda")
        ops.add_group_normed(r, None if delta is None else delta[:rows].cuda(), None if delta is None else weight, groups, 1e-3, 0.5, out, rows,
                             next_weight=follow, next_groups=groups, next_eps=1e-2)
        got[rows] = r[:64].cpu(), out[:64].cpu()
    assert torch.equal(got[64][0], got[130][0]) and torch.equal(got[64][1], got[130][1])


@pytest.mark.parametrize("rows,D,Dx", [(3, 100, 129), (70, 2048, 2049), (3, 511, 4100), (1, 1, 1)])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_gated_add(rows, D, Dx, dtype):
    from hector_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(D)
    a, b, x = (torch.randn(rows, n, generator=g).to(dtype) for n in (D, D, Dx))
    gate = torch.randn(Dx, generator=g).to(dtype) * Dx ** -0.5
    out = torch.empty(rows, D, dtype=dtype, device="cuda")
    ops.gated_add(out, a.cuda(), b.cuda(), x.cuda(), gate.cuda(), rows)
    close(out, a.to(F64) + torch.sigmoid((x.to(F64) * gate.to(F64)).sum(-1, keepdim=True)) * b.to(F64), dtype)


@pytest.mark.parametrize("rows,W", [(3, 1), (70, 511), (3, 8192), (3, 8193), (70, 2049)])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_polynorm(rows, W, dtype):
    from hector_engine_amd.kernels import ops
    x = torch.randn(rows, W, generator=torch.Generator().manual_seed(W)).to(dtype)
    numbers, z = torch.tensor([0.5, -0.3, 0.2, 0.1]), x.to(F64)
    out = torch.empty(rows, W, dtype=dtype, device="cuda")
    ops.polynorm(out, x.cuda(), numbers.cuda(), rows, 1e-3)
    a, b, c, e = numbers.to(F64).tolist()
    close(out, a * gn(z, 1, 1e-3) + b * gn(z * z, 1, 1e-3) + c * gn(z ** 3, 1, 1e-3) + e, dtype)
    same = x.cuda()                    # in place
    ops.polynorm(same, same, numbers.cuda(), rows, 1e-3)
    assert torch.equal(same, out)
