"""bf16 products of many rows in tiles, and the experts of a routed feed-forward over the rows that chose them."""
import pytest
import torch

from hector_engine_amd.kernels import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(BF16)


# fp32 sums of bf16 products in another order: a few ulp of 32 bits of the sum of magnitudes, then one rounding to bf16
def near(got, want, size, bf16):
    tol = 1e-6 * size + (2 ** -8 * want.abs() if bf16 else 0)
    assert ((got.double().cpu() - want).abs() <= tol + 1e-30).all()


@pytest.mark.parametrize("bm", [128, 256])
@pytest.mark.parametrize("M,N,K", [(1, 4, 64), (128, 256, 128), (127, 260, 192), (257, 516, 64), (300, 12, 320), (2200, 300, 64)])
def test_products_in_tiles(bm, M, N, K):
    x, w, b = rnd(M, K, seed=1), rnd(N, K, seed=2), rnd(N, seed=3)
    want = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    out = torch.full((M + 1, N), 7.0, dtype=BF16, device="cuda")
    ops.gemm_tall(out, x.cuda(), w.cuda(), b.cuda(), M, bm=bm)
    near(out[:M], want + b.double(), size + b.double().abs(), True)
    assert (out[M] == 7).all()
    out = torch.full((M + 1, N), 7.0, device="cuda")
    ops.gemm_tall(out, x.cuda(), w.cuda(), None, M, bm=bm)
    near(out[:M], want, size, False)
    assert (out[M] == 7).all()
    for act in ((1.0, 0.0, 0.0, 0.0), (1.702, 2.0, 1.0, 0.0)):
        out = torch.full((M + 1, N // 2), 7.0, dtype=BF16, device="cuda")
        ops.gemm_tall(out, x.cuda(), w.cuda(), None, M, bm=bm, act=act)
        g, u = want[:, 0::2], want[:, 1::2]
        if act[1]:
            g, u = g.clamp(max=act[1]), u.clamp(-act[1], act[1])
        gated = g * torch.sigmoid(act[0] * g) * (u + act[2])
        # the derivatives of the activation are at most 1.2 (|u| + 1) and |g| + 1
        # and gate and up are rounded to bf16 before it
        slack = 2 ** -8 * (want[:, 0::2].abs() * 1.2 * (u.abs() + 1) + want[:, 1::2].abs() * (g.abs() + 1))
        got, bound = out[:M].double().cpu(), 1e-6 * (size[:, 0::2] * 1.2 * (u.abs() + 1) + size[:, 1::2] * (g.abs() + 1))
        assert ((got - gated).abs() <= bound + slack + 2 ** -8 * gated.abs()).all()
        assert (out[M] == 7).all()


TILES = [(256, 256), (256, 224), (256, 192), (256, 160), (128, 288), (128, 256), (128, 224), (128, 160)]


# one stage and fewer stages than the rings hold; a single output, edges of tiles, rows of results that begin at no 16-byte boundary,
# more tiles than the chip has units (a workgroup goes from tile to tile), rows and columns of tiles that do not divide by the band
@pytest.mark.parametrize("M,N,K", [(1, 4, 64), (255, 156, 64), (257, 452, 128), (130, 300, 320), (1300, 4600, 64), (2500, 6404, 192)])
@pytest.mark.parametrize("bm,bn", TILES)
def test_every_tile(bm, bn, M, N, K):
    x, w, b = rnd(M, K, seed=1).cuda(), rnd(N, K, seed=2).cuda(), rnd(N, seed=3).cuda()
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    out = torch.full((M + 1, N), 7.0, dtype=BF16, device="cuda")
    for bias in (None, b):
        ops.gemm_tall(out, x, w, bias, M, bm=bm, bn=bn)
        plus = 0 if bias is None else bias.double()
        near(out[:M], (want + plus).cpu(), (size + abs(plus)).cpu(), True)
        assert (out[M] == 7).all()
    act = (1.0, 0.0, 0.0, 0.0)
    gated = torch.full((M + 1, N // 2), 7.0, dtype=BF16, device="cuda")
    ops.gemm_tall(gated, x, w, None, M, bm=bm, bn=bn, act=act)
    ops.gemm_tall(out, x, w, None, M, bm=bm, bn=bn)
    two = torch.empty(M, N // 2, dtype=BF16, device="cuda")
    ops.silu_mul(two, out, M, True)            # the activation of the rounded products, by the kernel that reads them from memory
    assert torch.equal(gated[:M], two)         # (the same function of the same bf16 gates and ups)
    assert (gated[M] == 7).all()


@pytest.mark.parametrize("act", [(1.0, 0.0, 0.0, 0.0), (1.702, 7.0, 1.0, 0.0)])
def test_the_gate_of_the_epilogue(act):
    """Every bf16 gate there is, infinities and NaN among them, beside ups of all sizes: the bits of the kernel that reads gate and up from memory."""
    gates = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(BF16).cuda()
    ups = torch.cat([rnd(60, seed=5), torch.tensor([0.0, -0.0, 1e-38, 3e38, -3e38]).to(BF16)]).cuda()
    N, M, K = 65536, 65, 64
    x, w = torch.zeros(M, K, dtype=BF16, device="cuda"), torch.zeros(2 * N, K, dtype=BF16, device="cuda")
    x[:, 0], x[:, 1], w[0::2, 0], w[1::2, 1] = 1.0, ups, gates, 1.0          # (row m, column n: gate n, up m, and products with zero)
    product = torch.empty(M, 2 * N, dtype=BF16, device="cuda")
    ops.gemm_tall(product, x, w, None, M)
    one, two = (torch.empty(M, N, dtype=BF16, device="cuda") for _ in range(2))
    ops.gemm_tall(one, x, w, None, M, act=act)
    ops.silu_mul(two, product, M, True, alpha=act[0], limit=act[1], up_shift=act[2])
    assert product[:, 0::2].isinf().any(0).sum() == 2 and product[:, 0::2].isnan().any(0).sum() == 254
    assert torch.equal(one.isnan(), two.isnan()) and torch.equal(one.nan_to_num(7.0), two.nan_to_num(7.0))


@pytest.mark.parametrize("bm", [128, 256])
@pytest.mark.parametrize("consts", [{}, {"alpha": 1.702, "limit": 1.5, "up_shift": 1.0}])
def test_the_experts_activations_are_those_behind_the_product_over_all_of_them(bm, consts):
    """Bit for bit: the router of a later layer may read rows that no norm has evened out, and there a last bit becomes another choice."""
    rows, real, top, D, I = 600, 16, 4, 128, 512
    x, gate_up = rnd(rows, D, seed=11).cuda(), rnd(2 * real * I, D, seed=12, scale=0.2).cuda()
    g = torch.Generator().manual_seed(13)
    ids = torch.stack([torch.randperm(real, generator=g)[:top] for _ in range(rows)]).int().cuda()
    weights = torch.rand(rows, top, generator=g).cuda()
    dense = torch.zeros(rows, real + 1, device="cuda").scatter_(1, ids.long(), weights)
    product, want = torch.empty(rows, 2 * real * I, dtype=BF16, device="cuda"), torch.empty(rows, real * I, dtype=BF16, device="cuda")
    ops.gemm_tall(product, x, gate_up, None, rows)
    ops.routed_act(want, product, dense, None, rows, real, I, **consts)
    lists = torch.empty(ops.routed_groups_sizes(rows, top, real, bm)[0], dtype=torch.int32, device="cuda")
    got = torch.zeros_like(want)
    ops.routed_groups_act(got, lists, x, gate_up, ids, weights, rows, real, I, bm=bm, **consts)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,N,K,slices", [(70, 300, 128, 2), (203, 460, 1536, 8), (257, 2052, 768, 4)])
@pytest.mark.parametrize("bm,bn", TILES)
def test_k_slices(bm, bn, M, N, K, slices):
    """Each slice is the product of its stretch of K, bit for bit."""
    x, w = rnd(M, K, seed=1).cuda(), rnd(N, K, seed=2).cuda()
    out = torch.full((slices, M, N), 7.0, device="cuda")
    ops.gemm_tall(out, x, w, None, M, bm=bm, bn=bn, slices=slices)
    for s in range(slices):
        part, alone = slice(s * K // slices, (s + 1) * K // slices), torch.empty(M, N, device="cuda")
        ops.gemm_tall(alone, x[:, part].contiguous(), w[:, part].contiguous(), None, M, bm=bm, bn=bn)
        assert torch.equal(out[s], alone)


@pytest.mark.parametrize("bm", [128, 256])
@pytest.mark.parametrize("rows,real,identity,top", [(1, 3, 0, 1), (130, 5, 1, 2), (300, 16, 2, 4), (513, 1, 0, 1), (700, 40, 0, 8)])
def test_experts_over_the_rows_that_chose_them(bm, rows, real, identity, top):
    D, I = 128, 192
    x = rnd(rows, D, seed=5)
    gate_up, down = rnd(2 * real * I, D, seed=6, scale=0.2), rnd(D, real * I + (D if identity else 0), seed=7, scale=0.2)
    g = torch.Generator().manual_seed(8)
    ids = torch.stack([torch.randperm(real + identity, generator=g)[:top] for _ in range(rows)]).int()
    ids[rows // 2:, 0] = 0 if real > 1 and top == 1 else ids[rows // 2:, 0]          # an expert with many rows, others with few
    ids[0, top - 1] = -1                                                             # a choice that found nothing
    weights = torch.rand(rows, top, generator=g)
    weights[ids < 0] = 0
    dense = torch.zeros(rows, real + 1)
    for k in range(top):
        for e in range(real):
            dense[:, e] += weights[:, k] * (ids[:, k] == e)
        dense[:, real] += weights[:, k] * (ids[:, k] >= real)
    ints, slots = ops.routed_groups_sizes(rows, top, real, bm)
    out = torch.full((rows, D), 7.0, dtype=BF16, device="cuda")
    h = torch.full((slots, I), float("nan"), dtype=BF16, device="cuda")
    ops.routed_groups(out, torch.full((ints,), -5, dtype=torch.int32, device="cuda"), h,
                      torch.full((slots, D), float("nan"), device="cuda"), x.cuda(), gate_up.cuda(), down.cuda(), ids.cuda(),
                      weights.cuda(), dense.cuda(), rows, real, I, bm=bm)
    want, size = torch.zeros(rows, D, dtype=torch.float64), torch.zeros(rows, D, dtype=torch.float64)
    for e in range(real):
        gu = x.double() @ gate_up[2 * e * I:2 * (e + 1) * I].double().T
        a = gu[:, 0::2] * torch.sigmoid(gu[:, 0::2]) * gu[:, 1::2] * dense[:, e:e + 1].double()
        d = down[:, e * I:(e + 1) * I].double()
        want += a @ d.T
        size += a.abs() @ d.abs().T
    if identity:
        want += dense[:, real:].double() * x.double()
        size += dense[:, real:].double() * x.double().abs()
    # gates and ups are rounded to bf16 (which moves an activation by 2.2 times its rounding at most here), the activations and the result too
    assert ((out.double().cpu() - want).abs() <= 2 ** -8 * 3.2 * size + 2 ** -8 * want.abs() + 1e-3).all()
    if not identity:
        # the activations alone, spread over the columns of all experts: what the second half read, zeros elsewhere
        wide = torch.zeros(rows, real * I, dtype=BF16, device="cuda")
        lists = torch.full((ints,), -5, dtype=torch.int32, device="cuda")
        ops.routed_groups_act(wide, lists, x.cuda(), gate_up.cuda(), ids.cuda(), weights.cuda(), rows, real, I, bm=bm)
        tile_rows = (real + 1 + 3) // 4 * 4
        rows_of = lists[tile_rows:tile_rows + slots].cpu()
        begin = lists[:real + 1].cpu()
        for e in range(real):
            for slot in range(int(begin[e]) * bm, int(begin[e + 1]) * bm):
                if rows_of[slot] >= 0:
                    assert torch.equal(wide[rows_of[slot], e * I:(e + 1) * I], h[slot])
                    wide[rows_of[slot], e * I:(e + 1) * I] = 0
        assert (wide == 0).all()


def test_experts_sums_lie_by_choice():
    """partial holds a row a choice, whatever the slots of the tiles: nothing is written behind it, and the two sizes give the same bits."""
    rows, real, top, D, I, bm = 70, 40, 2, 128, 64, 128
    x, gate_up, down = rnd(rows, D, seed=1).cuda(), rnd(2 * real * I, D, seed=2, scale=0.2).cuda(), rnd(D, real * I, seed=3, scale=0.2).cuda()
    g = torch.Generator().manual_seed(4)
    ids = torch.stack([torch.randperm(real, generator=g)[:top] for _ in range(rows)]).int().cuda()
    weights = torch.rand(rows, top, generator=g).cuda()
    dense = torch.zeros(rows, real + 1, device="cuda").scatter_(1, ids.long(), weights)
    ints, slots = ops.routed_groups_sizes(rows, top, real, bm)
    assert slots > 20 * rows * top
    h = torch.empty(slots, I, dtype=BF16, device="cuda")
    room = torch.full((rows * top + 1, D), 7.0, device="cuda")
    outs = []
    for partial in (room[:rows * top], torch.full((slots, D), float("nan"), device="cuda")):
        outs.append(torch.empty(rows, D, dtype=BF16, device="cuda"))
        ops.routed_groups(outs[-1], torch.empty(ints, dtype=torch.int32, device="cuda"), h, partial, x, gate_up, down, ids, weights,
                          dense, rows, real, I, bm=bm)
    assert torch.equal(*outs) and (room[-1] == 7).all() and not (room[:-1] == 7).all(1).any()
