"""A token's choice among 1 to 1024 outputs: every count of outputs a lane holds, ties, outputs that are masked or always kept."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def choice(c, groups, keep, top):
    """The outputs chosen from the scores c (a list) by the stated order; -1 where none is left."""
    size = len(c) // groups
    best = [max(c[g * size:(g + 1) * size]) for g in range(groups)]
    kept = {g for g in range(groups) if best[g] == math.inf}
    kept |= set(sorted((g for g in range(groups) if g not in kept), key=lambda g: (-best[g], g))[:keep])
    c = [v if keep >= groups or e // size in kept else -math.inf for e, v in enumerate(c)]
    return sorted(range(len(c)), key=lambda e: (-c[e], e))[:top]


@pytest.mark.parametrize("E,real,groups,keep,top", [(1, 1, 1, 1, 1), (18, 16, 3, 2, 4), (63, 60, 7, 3, 27), (64, 64, 64, 9, 9), (65, 60, 5, 1, 13),
                                                    (256, 250, 1, 1, 16), (257, 200, 257, 200, 100), (1024, 1000, 8, 3, 8)])
@pytest.mark.parametrize("normalize", [False, True])
def test_choice(E, real, groups, keep, top, normalize):
    from hector_engine_amd.kernels import ops
    rows = 5
    logits = torch.randn(rows, E, generator=torch.Generator().manual_seed(E))
    logits[1] = logits[1].round()                              # ties in the score
    # the correction decides: multiples of 1/8 from -3 on, far apart beside the scores' rounding, with ties, masked and kept outputs
    correction = torch.arange(E).mul(37).remainder(max(3, E // 2)).float() / 8 - 3
    correction[E // 3:E // 3 + E // 7] = -math.inf
    if E > 4:
        correction[E - 2] = math.inf
    for corr in (None, correction):
        dense = torch.full((rows, real + 1), math.nan, device="cuda")
        ids, weights = torch.full((rows, top), 77, dtype=torch.int32, device="cuda"), torch.full((rows, top), math.nan, device="cuda")
        ops.route_tokens(dense, ids, weights, logits.cuda(), None if corr is None else corr.cuda(), rows, real, groups, keep, top, 1.5, normalize=normalize)
        s = torch.softmax(logits.double(), -1)
        for r in range(rows):
            c = logits[r].tolist() if corr is None else (torch.softmax(logits[r], -1) + corr).tolist()
            got = ids[r].tolist()
            if corr is None:
                assert got == choice(c, groups, keep, top)
            else:       # (scores of two outputs with one correction may round to a tie, or out of one: the corrections are the ones of the order)
                want = choice(c, groups, keep, top)
                assert sorted(set(got)) == sorted(got) and [corr[e] for e in got] == [corr[e] for e in want]
            w = s[r, got] * 1.5
            if normalize:
                w = w / s[r, got].sum()
            # fp32 exponentials, sums of up to 1024 of them and of up to 100 scores: some 1e-6
            assert torch.allclose(weights[r].cpu().double(), w, rtol=4e-6, atol=1e-9)
            want = torch.zeros(real + 1, dtype=torch.float64)
            for e, v in zip(got, w):
                want[min(e, real)] += v
            assert torch.allclose(dense[r].cpu().double(), want, rtol=4e-6, atol=1e-9)


def _routed(ops, x, router, rows, groups, keep, top, **more):
    E = router.shape[0]
    dense = torch.full((rows, E - 1), math.nan, device="cuda")
    ids, weights = torch.full((rows, top), 77, dtype=torch.int32, device="cuda"), torch.full((rows, top), math.nan, device="cuda")
    ops.route_tokens(dense, ids, weights, None, None, rows, E - 2, groups, keep, top, 1.5, x=x, router=router, **more)
    return dense, ids, weights


@pytest.mark.parametrize("E,D,groups,keep,top", [(3, 4, 1, 1, 2), (18, 2048, 3, 2, 4), (64, 260, 8, 2, 5), (100, 1028, 1, 1, 8), (300, 64, 5, 3, 9),
                                                 (18, 42, 1, 1, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_that_share_a_workgroup(E, D, groups, keep, top, dtype):
    """Steps of more than 256 rows read the router's rows once for two rows: each row's result has the bits it has alone."""
    from hector_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(D)
    for rows in (257, 518):
        x = torch.randn(rows, D, generator=g).to(dtype).cuda()
        router = torch.randn(E, D, generator=g).cuda()
        got = _routed(ops, x, router, rows, groups, keep, top, normalize=True)
        at = 0
        for n in (1, 200, 56, rows - 257):
            if n == 0:
                continue
            alone = _routed(ops, x[at:at + n].clone(), router, n, groups, keep, top, normalize=True)
            for a, b in zip(got, alone):
                assert torch.equal(a[at:at + n], b)
            at += n
        assert at == rows


@pytest.mark.parametrize("rows,E,D,count,pieces", [(1, 18, 2048, 256, True), (3, 64, 8, 1, False), (16, 5, 520, 65, True), (300, 33, 264, 7, False)])
def test_the_norms_scale_with_the_choice(rows, E, D, count, pieces):
    """Rows whose norm's scale is owed: the launch gives the rows and the choice of the two launches it stands for, bit for bit."""
    from hector_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, D, generator=g).bfloat16().cuda()
    partials = (torch.rand(rows, count, generator=g) * D / count).cuda()
    router = torch.randn(E, D, generator=g).cuda()
    given = x.view(rows, D // 8, 8).transpose(0, 1).contiguous() if pieces else x
    want_rows, got_rows = torch.empty_like(x), torch.full_like(x, math.nan)
    ops.scale_rows(want_rows, given, partials, 1e-6, rows, pieces)
    want = _routed(ops, want_rows, router, rows, 1, 1, 3)
    got = _routed(ops, given, router, rows, 1, 1, 3, x_pieces=pieces, owed=(partials, 1e-6, got_rows))
    assert torch.equal(got_rows, want_rows)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    with pytest.raises(RuntimeError):
        ops.route_tokens(*want, None, None, rows, E - 2, 1, 1, 3, 1.5, x=given, router=torch.randn(65, D, device="cuda"), x_pieces=pieces,
                         owed=(partials, 1e-6, got_rows))


@pytest.mark.parametrize("E,D,count", [(3, 2040, 257), (18, 2048, 255), (17, 2056, 600), (41, 1032, 256), (9, 4104, 1)])
@pytest.mark.parametrize("pieces", [False, True])
def test_a_routers_turns_and_parts_at_their_edges(E, D, count, pieces):
    """Rows around whole turns of loads, scales of more parts than are asked for ahead, biases and corrections: the bits of the same
    rows scaled beforehand and routed two a workgroup."""
    from hector_engine_amd.kernels import ops
    g, rows = torch.Generator().manual_seed(D + E), 2
    x = torch.randn(rows, D, generator=g).bfloat16().cuda()
    partials = (torch.rand(rows, count, generator=g) * D / count).cuda()
    router, bias, correction = (torch.randn(*s, generator=g).cuda() for s in ((E, D), (E,), (E,)))
    given = x.view(rows, D // 8, 8).transpose(0, 1).contiguous() if pieces else x
    scaled, got_rows = torch.empty_like(x), torch.full_like(x, math.nan)
    ops.scale_rows(scaled, given, partials, 1e-6, rows, pieces)

    def route(x, n, **more):
        dense, ids = torch.full((n, E + 1), math.nan, device="cuda"), torch.full((n, 3), 77, dtype=torch.int32, device="cuda")
        weights = torch.full((n, 3), math.nan, device="cuda")
        ops.route_tokens(dense, ids, weights, None, correction, n, E, 1, 1, 3, 1.5, x=x, router=router, bias=bias, **more)
        return dense, ids, weights
    want = route(scaled.repeat(150, 1), 150 * rows)
    got = route(given, rows, x_pieces=pieces, owed=(partials, 1e-6, got_rows))
    assert torch.equal(got_rows, scaled)
    for a, b in zip(got, want):
        assert torch.equal(a, b[:rows]) and torch.equal(a, b[-rows:])


@pytest.mark.parametrize("copies", [2, 4, 12])
@pytest.mark.parametrize("rows", [40, 300])
def test_equal_outputs_tie_wherever_they_stand(copies, rows):
    """Outputs with one score and one correction, 64 apart: a lane's first output among them, whose correction is asked for ahead. The scores meet
    the corrections in two roundings, so that the copies tie and are chosen in the order of their numbers; from logits and from rows."""
    from hector_engine_amd.kernels import ops
    g, E, D, top = torch.Generator().manual_seed(copies), 64 * copies, 256, 3 * copies
    correction = (0.1 * torch.randn(64, generator=g)).repeat(copies).cuda()
    x, router = torch.randn(rows, D, generator=g).bfloat16().cuda(), (0.1 * torch.randn(64, D, generator=g)).repeat(copies, 1).cuda()
    logits = torch.randn(rows, 64, generator=g).repeat(1, copies).cuda()
    for given in (dict(logits=logits), dict(logits=None, x=x, router=router)):
        dense, ids = torch.empty(rows, E + 1, device="cuda"), torch.full((rows, top), 77, dtype=torch.int32, device="cuda")
        ops.route_tokens(dense, ids, torch.empty(rows, top, device="cuda"), given.pop("logits"), correction, rows, E, 1, 1, top, 1.0, **given)
        assert torch.equal(ids, torch.cat([ids[:, i * copies:i * copies + 1] + 64 * torch.arange(copies, device="cuda", dtype=torch.int32) for i in range(3)], 1))


@pytest.mark.parametrize("rows,top,real,I,D,shared", [(1, 4, 16, 64, 128, 32), (2, 4, 16, 520, 264, 0), (5, 3, 30, 72, 1032, 40), (16, 4, 128, 24, 64, 8), (17, 4, 140, 24, 64, 8), (33, 2, 140, 16, 72, 16)])
@pytest.mark.parametrize("kind", ["apart", "same", "some", "none"])
def test_chosen_experts_of_a_row_do_not_depend_on_the_others(rows, top, real, I, D, shared, kind):
    """Experts that one row chose, several, or all, ids that name no expert, up to 64 ids and more of them: each row has the bits it has alone,
    whichever way its weights come."""
    from hector_engine_amd.kernels import ops
    g = torch.Generator().manual_seed(rows + I)
    ids = torch.stack([torch.randperm(real, generator=g)[:top] for _ in range(rows)])
    if kind == "apart":
        ids = torch.randperm(real, generator=g)[:rows * top].view(rows, top)
    elif kind == "same":
        ids[:] = ids[0].clone()
    elif kind == "none":
        ids[::2, 0], ids[1::3, top - 1] = real, -1
    ids, weights = ids.int().contiguous().cuda(), torch.rand(rows, top, generator=g).cuda()
    x, dense = torch.randn(rows, D, generator=g).bfloat16().cuda(), torch.zeros(rows, real + 1, device="cuda")
    gate_up, down = ((0.1 * torch.randn(*s, generator=g)).bfloat16().cuda() for s in ((2 * (real * I + shared), D), (D, real * I + shared)))

    def run(at):
        n = at.stop - at.start
        out, h = torch.full((n + 1, D), 7.0, dtype=torch.bfloat16, device="cuda"), torch.empty(n * (top * I + shared), dtype=torch.bfloat16, device="cuda")
        ops.chosen_experts(out, h, x[at].contiguous(), gate_up, down, ids[at].contiguous(), weights[at].contiguous(), dense[at].contiguous(), n, real, I, shared=shared)
        assert (out[n] == 7).all()
        return out[:n]
    whole = run(slice(0, rows))
    assert whole.abs().max() > 0
    for r in range(rows):
        assert torch.equal(run(slice(r, r + 1))[0], whole[r])
