"""The order in which the products of few rows add up, and what they leave out without changing it.

The order is told with the tile kernel, which adds in the order of k: K is laid out anew in the order of units of 64 k that is stated for the kernel under
test, 16 of a unit's k to a lane group as that has them, and the results are the same bits, which another order's are not."""
from types import SimpleNamespace

import pytest
import torch

from hector_engine_amd.engine.scratch import ScratchPool
from hector_engine_amd.kernels import ops
from hector_engine_amd.parts.base import BuildEnv
from hector_engine_amd.parts.linear import Linear

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def laid_out(t):
    """[rows, K] as [rows, units, 64], a unit's k in the order the tile kernel needs to multiply the same ones together: a lane group has 16
    neighbouring k, 8 to an instruction, there the 8 of each half of the unit."""
    rows, K = t.shape
    units = -(-K // 64)
    whole = torch.zeros(rows, units * 64, dtype=t.dtype, device=t.device)
    whole[:, :K] = t
    return whole.view(rows, units, 4, 2, 8).transpose(2, 3).reshape(rows, units, 64)


def chain(xu, wu, order):
    """The 32-bit sums over the units in `order`, one after the other."""
    M, N = len(xu), len(wu)
    out = torch.zeros(M, -(-N // 4) * 4, device="cuda")
    if len(order):
        x, w = xu[:, order].reshape(M, -1).contiguous(), torch.zeros(out.shape[1], 64 * len(order), dtype=BF16, device="cuda")
        w[:N] = wu[:, order].reshape(N, -1)
        ops.gemm_tall(out, x, w, None, M)
    return out[:, :N]


def chained(xu, wu, block, order_of, turns):
    """The same where the order depends on the workgroup (block [N]: a weight row's): order_of(turn) for each of `turns` [workgroups]."""
    out = torch.empty(len(xu), len(wu), device="cuda")
    turn = turns[block]
    for t in turn.unique().tolist():
        rows = (turn == t).nonzero()[:, 0]
        out[:, rows] = chain(xu, wu[rows], order_of(t))
    return out


def operands(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(N + M)
    return (torch.randn(*s, generator=g, device="cuda").to(BF16) for s in ((M, K), (N, K)))


# (a shape for each branch of the ordered tiling, on 256 units: weight rows a workgroup has, its wavefronts, units of a turn)
ORDERED = [(3, 65536, 2048, 32, 8, 2), (12, 65537, 2048, 64, 4, 4), (5, 896, 8192, 4, 8, 2), (4, 300, 8256, 16, 8, 2), (16, 10240, 8192, 64, 4, 4),
           (8, 4608, 8192, 18, 8, 2), (2, 10240, 8192, 20, 8, 2), (4, 8192, 16384, 32, 8, 4), (1, 8192, 8192, 32, 4, 8), (7, 16384, 3584, 32, 4, 4),
           (4, 16384, 5120, 32, 8, 2), (9, 16500, 5120, 64, 8, 2), (4, 4608, 3584, 18, 8, 8), (1, 3584, 5128, 14, 8, 2), (4, 512, 520, 2, 4, 8),
           (20, 4608, 3584, 18, 8, 2), (17, 3584, 18944, 14, 4, 2), (32, 16384, 3584, 32, 4, 4), (24, 65537, 2048, 32, 4, 4), (31, 4104, 8200, 18, 4, 4),
           (29, 300, 1032, 16, 8, 2)]


@pytest.mark.parametrize("M,N,K,rows,waves,turn", ORDERED)
def test_ordered_sums_are_added_as_they_always_were(M, N, K, rows, waves, turn):
    """Wavefronts with a K slice each, whose walk begins at a turn of the workgroup's own and goes around, and which are added in their order; an
    activation walks the same way. Above 16 rows that is the only order."""
    if ops.compute_units() != 256:
        pytest.skip("the tilings of 256 compute units")
    x, w = operands(M, N, K)
    xu, wu = laid_out(x), laid_out(w)
    units, block, each = xu.shape[1], torch.arange(N, device="cuda") // rows, -(-(-(-K // waves)) // 64)
    want = torch.zeros(M, N, device="cuda")
    for v in range(waves):
        u0 = min(v * each, units)
        u1 = min(units, u0 + each)
        whole = max(min(u1, K // 64) - u0, 0) // turn * turn
        starts = (3 * torch.arange(-(-N // rows), device="cuda")) % max(whole // turn, 1) * turn
        want = want + chained(xu, wu, block, lambda f: [u0 + (f + j) % whole for j in range(whole)] + list(range(u0 + whole, u1)), starts)
    pieces = x.view(M, K // 8, 8).transpose(0, 1).contiguous()
    for given, more in ((x, {}), (pieces, dict(x_pieces=True)))[:2 if M <= 16 else 1]:
        out = torch.empty(M, N, device="cuda")
        ops.gemm_blocksplit(out, given, w, None, M, ordered=M <= 16, **more)
        assert torch.equal(out, want)
    half = torch.empty(M, N, dtype=BF16, device="cuda")
    ops.gemm_blocksplit(half, x, w, None, M, ordered=M <= 16, unary="relu")
    assert torch.equal(half, want.to(BF16).relu())
    if M > 16:
        return
    free = torch.empty(M, N, device="cuda")
    ops.gemm_blocksplit(free, x, w, None, M)
    assert not torch.equal(free, want)                        # (another order does give other bits)


@pytest.mark.parametrize("M,N,K,R,NWV", [(17, 4608, 3584, 1, 8), (64, 4608, 3584, 1, 8), (33, 3584, 18944, 1, 8), (20, 900, 1032, 1, 4), (64, 16400, 1096, 1, 16),
                                         (32, 16400, 1032, 1, 8), (24, 65600, 320, 2, 8), (40, 65600, 576, 1, 16)])
def test_products_of_17_to_64_rows_are_added_as_they_always_were(M, N, K, R, NWV):
    """K slices of whole chunks of 128 k, each walked from a chunk of the workgroup's own on and around."""
    if ops.compute_units() != 256:
        pytest.skip("the tilings of 256 compute units")
    x, w = operands(M, N, K)
    xu, wu = laid_out(x), laid_out(w)
    groups, slices = ops.gemm_rows_plan(M, N, K)
    rows = 16 * R * NWV
    if N >= 16384:
        slots = 256 * (1 if NWV == 16 or R == 2 else 2)
        rounds = -(-N // (slots * rows))
        rows = min(rows, (-(-N // (slots * rounds)) + 3) // 4 * 4)
    assert groups == -(-N // rows)
    wanted = 1
    while groups * wanted < 192 and K // (2 * wanted) >= 256 and wanted < 32:
        wanted *= 2
    each = -(-(-(-K // wanted)) // 128) * 128
    assert slices == -(-K // each)
    block, want = torch.arange(N, device="cuda") // rows, []
    for s in range(slices):
        k0, k1 = s * each, min(K, (s + 1) * each)
        chunks, last = -(-(k1 - k0) // 128), -(-k1 // 64)
        starts = (5 * torch.arange(groups, device="cuda")) % chunks
        want.append(chained(xu, wu, block, lambda r: [u for c in range(chunks) for u in (k0 // 64 + 2 * ((r + c) % chunks), k0 // 64 + 2 * ((r + c) % chunks) + 1)
                                                      if u < last], starts))
    if slices == 1:
        out = torch.empty(M, N, device="cuda")
        ops.gemm_rows(out, None, x, w, None, M)
        assert torch.equal(out, want[0])
    else:
        partial = torch.empty(slices, M, N, device="cuda")
        ops.gemm_rows(None, partial, x, w, None, M)
        assert torch.equal(partial, torch.stack(want))


def used_case(M, count, size, extra, N, K, along_k, seed):
    g = torch.Generator().manual_seed(seed)
    used = torch.rand(M, count + 1, generator=g) * (torch.rand(M, count + 1, generator=g) < 1.5 / count)
    used[0, count // 2] = 0.5
    x, w = (0.5 * torch.randn(M, K, generator=g)).to(BF16), (0.05 * torch.randn(N, K, generator=g)).to(BF16).cuda()
    if along_k:
        for e in range(count):
            x[:, e * size:(e + 1) * size] *= (used[:, e] != 0)[:, None]
    return used.cuda(), (used[:, :count] != 0).any(0).tolist(), x.cuda(), w


@pytest.mark.parametrize("M", [1, 4, 7, 16])
@pytest.mark.parametrize("pieces", [False, True])
@pytest.mark.parametrize("N,count,size,extra", [(2048, 16, 2048, 0), (320, 5, 512, 192), (4608, 3, 640, 0), (10240, 4, 2048, 0), (1024, 6, 1000, 0), (70000, 2, 576, 0)])
def test_ordered_products_leave_out_groups_along_k(M, pieces, N, count, size, extra):
    """The walk that begins at a turn of its own skips the turns of groups nobody uses: the bits of the whole product."""
    K = count * size + extra
    used, some, x, w = used_case(M, count, size, extra, N, K, True, N + M)
    given = x.view(M, K // 8, 8).transpose(0, 1).contiguous() if pieces else x
    whole, out = (torch.full((M + 1, N), 7.0, dtype=BF16, device="cuda") for _ in range(2))
    ops.gemm_blocksplit(whole, given, w, None, M, x_pieces=pieces, ordered=True)
    for nan in (False, True):
        if nan and size < 1024:                               # (a turn of a wavefront may meet two groups there)
            break
        for e in range(count):
            if nan and not some[e]:
                w[:, e * size:(e + 1) * size] = float("nan")
        ops.gemm_blocksplit(out, given, w, None, M, x_pieces=pieces, ordered=True, used=(used, count, size, True))
        assert torch.equal(out, whole) and (out[M] == 7).all()


@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("K,count,size,extra", [(2048, 16, 4096, 0), (520, 5, 300, 40), (64, 40, 16, 0), (1024, 3, 2, 6)])
def test_ordered_products_leave_out_groups_of_rows(M, K, count, size, extra):
    N = count * size + extra
    used, some, x, w = used_case(M, count, size, extra, N, K, False, N + M)
    whole, out = (torch.full((M, N), 7.0, dtype=BF16, device="cuda") for _ in range(2))
    ops.gemm_blocksplit(whole, x, w, None, M, ordered=True)
    ops.gemm_blocksplit(out, x, w, None, M, ordered=True, used=(used, count, size, False))
    for e in range(count):
        cols = slice(e * size, (e + 1) * size)
        assert torch.equal(out[:, cols], whole[:, cols]) if some[e] else ((out[:, cols] == whole[:, cols]) | (out[:, cols] == 7)).all()
    assert torch.equal(out[:, count * size:], whole[:, count * size:])
    if size >= 4096:
        assert (out == 7).all(0).sum() >= 0.9 * size * some.count(False)      # (a workgroup at a border computes both sides)


@pytest.mark.parametrize("M", [1, 3, 8, 16])
@pytest.mark.parametrize("pieces", [False, True])
@pytest.mark.parametrize("N,count,size,extra", [(2048, 16, 2048, 0), (320, 5, 512, 192), (4608, 3, 640, 0), (1032, 6, 1000, 0)])
def test_products_into_the_residual_rows_leave_out_groups_along_k(M, pieces, N, count, size, extra):
    """resid, the next norm's rows and their sums of squares have the bits they have with all weights read."""
    K = count * size + extra
    used, some, x, w = used_case(M, count, size, extra, N, K, True, N + M)
    given = x.view(M, K // 8, 8).transpose(0, 1).contiguous() if pieces else x
    r0, gain = torch.randn(M, N, device="cuda"), torch.rand(N, device="cuda").to(BF16)

    def left(**more):
        resid, xg = r0.clone(), torch.full(ops.pieces_shape(M, N) if pieces else (M, N), 7.0, dtype=BF16, device="cuda")
        sq = torch.full((M, ops.gemm_blocksplit_blocks(M, N, K)), float("nan"), device="cuda")
        ops.gemm_blocksplit(None, given, w, None, M, residual=(resid, gain, xg, sq), x_pieces=pieces, out_pieces=pieces, **more)
        return resid, xg, sq
    whole = left()
    for nan in (False, True):
        if nan and size < 1024:
            break
        for e in range(count):
            if nan and not some[e]:
                w[:, e * size:(e + 1) * size] = float("nan")
        assert all(torch.equal(a, b) for a, b in zip(left(used=(used, count, size, True)), whole))


@pytest.mark.parametrize("M,plan", [(4, (3, 0, 0)), (4, (0, 3, 0)), (8, (1, 8, 8)), (16, (4, 4, 0)), (8, (8, 1, 0)), (20, (4, 0, 0)), (20, (1, 4, 0)), (32, (3, 1, 0))])
def test_plans_of_no_tiling_are_refused(M, plan):
    x, w = torch.zeros(M, 512, dtype=BF16, device="cuda"), torch.zeros(64, 512, dtype=BF16, device="cuda")
    with pytest.raises(RuntimeError):
        ops.gemm_blocksplit(torch.empty(M, 64, device="cuda"), x, w, None, M, plan=plan)


def test_rows_beyond_32_bit_offsets_are_refused():
    """16 rows of 2^27 values, 4 GiB."""
    K = 1 << 27
    x, w = torch.empty(16, K, dtype=BF16, device="cuda"), torch.empty(2, K, dtype=BF16, device="cuda")
    with pytest.raises(RuntimeError):
        ops.gemm_blocksplit(torch.empty(16, 2, device="cuda"), x, w, None, 16)


@pytest.mark.parametrize("rows", [1, 16, 17])
def test_an_ordered_product_leaves_no_residual(rows):
    """A layer whose products keep their order gives its results as they are, also where the caller's stream would take them (above 16 rows
    there is one order)."""
    x, w = operands(rows, 512, 2048)
    lin = Linear(w)
    lin.ordered = True
    scratch = ScratchPool(torch.device("cuda:0"))
    ctx = SimpleNamespace(rows=rows, env=BuildEnv(torch.device("cuda:0"), BF16, True), scratch=scratch,
                          alloc=lambda shape, dtype=BF16: scratch.alloc(shape, dtype or BF16))
    resid = torch.zeros(rows, 512, device="cuda")
    norm = SimpleNamespace(carried=lambda: (torch.ones(512, dtype=BF16, device="cuda"), 1e-6))
    sink = SimpleNamespace(stream=SimpleNamespace(rows=rows, resid=resid, prepared=None), norm=norm, scale=1.0)
    out = lin(x, rows, ctx, sink=sink)
    if rows > 16:
        assert out is None and sink.stream.prepared is not None
        return
    want = torch.empty(rows, 512, dtype=BF16, device="cuda")
    ops.gemm_blocksplit(want, x, w, None, rows, ordered=True)
    assert torch.equal(out, want) and (resid == 0).all() and sink.stream.prepared is None
