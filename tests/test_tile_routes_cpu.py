"""Which products of many rows run through the tile kernels: the rules alone, over tensors without storage."""
import contextlib
import math
from types import SimpleNamespace

import pytest
import torch

from hector_engine_amd.kernels import ops, routes
from hector_engine_amd.parts.base import BuildEnv, PartSpec, build_part
from hector_engine_amd.parts.linear import Linear

BF16 = torch.bfloat16
CTX = SimpleNamespace(env=BuildEnv(torch.device("cpu"), BF16, True))


def empty(*shape, dtype=BF16):
    return torch.empty(shape, dtype=dtype, device="meta")


def experts(real=16, top=4, inter=2048, hidden=2048, **more):
    part = build_part("feed_forward", PartSpec("routed_experts", {
        "hidden_size": hidden, "intermediate_size": inter, "experts": real, "top": top, "correction": False, **more}), "m.", CTX.env)
    part.gate_up, part.down = Linear(empty(2 * real * inter, hidden)), Linear(empty(hidden, real * inter))
    return part


@contextlib.contextmanager
def route_before_the_library(takes):
    key = (BF16, BF16)
    routes.register_route("linear", key, "of_a_user", takes, lambda *a: None, before="library")
    try:
        yield
    finally:
        routes.unregister_route("linear", key, "of_a_user")


def test_a_registered_route_gets_the_gated_products_it_takes():
    lin, x = Linear(empty(9728, 896)), empty(700, 896)
    assert lin.tall_gated(700, CTX, x)
    with route_before_the_library(lambda c: c.N == 9728):
        assert not lin.tall_gated(700, CTX, x)
    with route_before_the_library(lambda c: c.N == 9720):
        assert lin.tall_gated(700, CTX, x)


@pytest.mark.parametrize("N", [2 * 16 * 2048, 2048])      # the experts' first product, their down product
def test_a_registered_route_gets_the_experts_products_it_takes(N):
    part, x = experts(), empty(2048, 2048)
    assert part._many_rows(2048, x, CTX)
    with route_before_the_library(lambda c: c.N == N):
        assert not part._many_rows(2048, x, CTX)


@pytest.mark.parametrize("N,K,tiles", [
    (9728, 896, {65: 0, 512: 0, 513: 128, 768: 128, 769: 0, 1207: 0, 1208: 256, 1536: 256, 1537: 0, 2048: 0, 12001: 0}),
    (8192, 1024, {512: 0, 640: 128, 1024: 128, 1025: 0, 1434: 256, 2048: 256, 2049: 0}),
    (1024, 256, {1000: 0, 4096: 0, 4992: 128, 8192: 128}),                # a few columns of tiles: units idle below
    (37888, 3584, {1024: 0, 1536: 0, 2048: 0, 2560: 0, 3072: 0}),         # a longer K: no relation to the sizes
    (4096, 2048, {2048: 0, 4096: 0}), (9728, 880, {600: 0}), (9724, 896, {600: 0})])
def test_which_gated_products_run_as_one_kernel(N, K, tiles):
    """At 256 units: tiles of 128 rows from 0.6 to 1 round of the chip, of 256 above that up to a round with 0.7 of it real."""
    lin = Linear(empty(N, K))
    assert {rows: lin.tall_gated(rows, CTX, empty(rows, K)) for rows in tiles} == tiles


def test_a_shared_expert_keeps_the_library_s_sums():
    """A router over rows that no norm has evened out turns last bits into other choices: a feed-forward beside it stays out."""
    def bound(kind, params):
        part = build_part("feed_forward", PartSpec(kind, params), "m.", CTX.env)
        part.bind({k: torch.zeros(v.shape, dtype=BF16) for k, v in part.tensor_specs().items()})
        return part
    mlp = {"hidden_size": 8, "intermediate_size": 16}
    assert bound("gated_mlp", mlp).down.one_round_tiles
    routed = bound("routed_experts", {**mlp, "experts": 4, "top": 2, "correction": False,
                                      "shared": {"gate": "sg", "feed_forward": PartSpec("gated_mlp", mlp)}})
    assert not routed.shared.down.one_round_tiles and not routed.down.one_round_tiles
    # one without a gate, and one that is itself routed and has a shared expert
    dense = PartSpec("dense_mlp", {**mlp, "activation": "relu2"})
    assert bound("dense_mlp", dense.params).up.one_round_tiles
    within = PartSpec("routed_experts", {**mlp, "experts": 4, "top": 2, "correction": False, "shared": {"gate": "sg", "feed_forward": dense}})
    for shared in (dense, within):
        part = bound("routed_experts", {**mlp, "experts": 4, "top": 2, "correction": False, "shared": {"feed_forward": shared}}).shared
        mlp_of = getattr(part, "shared", part)
        assert not mlp_of.up.one_round_tiles and not mlp_of.down.one_round_tiles


def test_k_slices_in_tiles_are_for_parts_that_allow_them(monkeypatch):
    """The experts' down product beside a shared expert is such a weight: its slices stay the library's, whose bits the tiles do not always give."""
    ran, N, K, rows = [], 3584, 18944, 200
    for module, name in ((ops, "gemm_tall"), (ops, "splitk_reduce"), (torch, "bmm")):
        monkeypatch.setattr(module, name, lambda *a, name=name, **k: ran.append(name))
    ctx = SimpleNamespace(env=CTX.env, alloc=lambda shape, dtype=BF16: empty(*shape, dtype=dtype))
    lin = Linear(empty(N, K))
    assert lin._library_slices(rows) == 8
    for allowed in (False, True):
        lin.one_round_tiles = allowed
        lin._library(empty(rows, K), None, rows, empty(rows, N), BF16, ctx)
    assert ran == ["bmm", "splitk_reduce", "gemm_tall", "splitk_reduce"]


@pytest.mark.parametrize("N,K,rows", [(3584, 18944, {65: True, 203: True, 257: True, 512: True}), (5120, 27648, {66: True, 380: True}),
                                      (2560, 14336, {97: False, 139: True, 262: True}),                  # half of the units
                                      (2048, 27648, {66: False, 128: False, 292: False}), (1024, 14336, {208: False}), (496, 27648, {78: False}),
                                      (3584, 18912, {203: False}), (3586, 18944, {203: False})])
def test_which_k_slices_run_in_tiles(N, K, rows):
    """At 256 units: more than 2048 columns, tiles for 0.7 of a round or more."""
    lin = Linear(empty(N, K))
    lin.one_round_tiles = True
    assert {r: lin._slices_in_tiles(r, lin._library_slices(r), empty(r, K)) for r in rows} == rows


def test_operands_the_tiles_do_not_read_stay_with_the_library():
    def shifted(*shape):
        return torch.empty(math.prod(shape) + 1, dtype=BF16)[1:].view(shape)
    for w, x in ((shifted(9728, 896), empty(600, 896)), (empty(9728, 896), shifted(600, 896))):
        assert Linear(w).tall_gated(600, CTX, x) == 0
    N, K, rows = 512, 16448, 12000
    for w, x, out in ((shifted(N, K), empty(rows, K), empty(rows, N)), (empty(N, K), empty(rows, K), shifted(rows, N)),
                      (empty(N, K), empty(rows, K), empty(rows, N))):
        lin = Linear(w)
        lin.one_round_tiles = True
        assert lin._long(rows, x, out, BF16) == (w.is_meta and out.is_meta)
    assert not experts()._many_rows(300, shifted(300, 2048), CTX)


def test_experts_beyond_the_tiles_offsets_stay_with_the_product_over_all():
    assert experts(real=512, inter=16320, hidden=64)._many_rows(4000, empty(4000, 64), CTX)
    assert not experts(real=512, inter=16384, hidden=64)._many_rows(4000, empty(4000, 64), CTX)


def test_many_experts_of_few_rows_take_no_more_scratch_than_the_product_over_all(monkeypatch):
    """An expert's tiles are mostly padding there: 65 rows that choose 8 of 256 experts, 33,280 slots for 520 choices."""
    part, rows, taken = experts(real=256, top=8, inter=2048, hidden=7168), 65, []

    def alloc(shape, dtype=BF16):
        taken.append(math.prod(shape) * dtype.itemsize)
        return empty(*shape, dtype=dtype)
    ctx = SimpleNamespace(env=CTX.env, alloc=alloc, scratch=SimpleNamespace(mark=lambda: None, release=lambda turn: None))
    x = empty(rows, 7168)
    bm = part._many_rows(rows, x, ctx)
    assert bm == 128
    monkeypatch.setattr(ops, "routed_groups", lambda *a, **k: None)
    part._by_expert(x, empty(rows, 257, dtype=torch.float32), empty(rows, 8, dtype=torch.int32), empty(rows, 8, dtype=torch.float32),
                    rows, bm, {}, ctx)
    assert sum(taken) <= rows * 3 * 256 * 2048 * 2       # gate and up of every expert, and their activations


@pytest.mark.parametrize("sizes,tiles", [
    (dict(real=16, top=4, inter=2048, hidden=2048), {65: 128, 512: 128, 768: 256, 2048: 256, 9000: 256}),
    (dict(real=64, top=4, inter=512, hidden=1024), {65: 128, 2048: 128, 4096: 256}),
    (dict(real=2, top=1, inter=64, hidden=1728), {65: 0, 224: 0, 1212: 0, 4096: 0}),      # small experts: two launches beat four
    (dict(real=256, top=128, inter=64, hidden=1152), {300: 0, 2948: 0, 4096: 0}),         # half of the experts, narrow tiles
    (dict(real=8, top=1, inter=4096, hidden=2048), {65: 0, 128: 0, 256: 128, 4096: 256})])  # few tiles of a long K
def test_which_routed_steps_run_expert_by_expert(sizes, tiles):
    """At 256 units: where the estimate of four launches over chosen rows is below 0.8 of the products over all experts."""
    part = experts(**sizes)
    assert {rows: part._many_rows(rows, empty(rows, sizes["hidden"]), CTX) for rows in tiles} == tiles


@pytest.mark.parametrize("sizes,left_out", [
    (dict(real=16, top=4, inter=2048, hidden=2048), {3: (True, True), 4: (True, True), 5: (False, True), 6: (False, False), 16: (False, False)}),
    (dict(real=16, top=4, inter=2048, hidden=768), {4: (False, True), 8: (False, False)}),       # short rows: the first product's check costs more
    (dict(real=40, top=4, inter=448, hidden=3072), {7: (True, False), 16: (False, False)}),      # groups of k shorter than a turn of the walk
    (dict(real=4, top=2, inter=1664, hidden=704), {2: (False, False), 11: (False, False)}),      # small weights; every expert chosen
    (dict(real=14, top=4, inter=2048, hidden=2048, identity_experts=2), {4: (False, True)})])
def test_which_steps_of_few_rows_leave_out_experts(monkeypatch, sizes, left_out):
    """Where the experts that nobody is expected to choose are enough bytes for what the check costs."""
    part, took = experts(**sizes), []

    class Product:
        weight = empty(8, 8)

        def own_tiles(self, rows, ctx):
            return False

        def __call__(self, x, rows, ctx, sink=None, used=None):
            took.append(used is not None and used[1:])
    part.router, part.gate_up, part.down = empty(18, sizes["hidden"], dtype=torch.float32), Product(), Product()
    for name in ("route_tokens", "routed_act"):
        monkeypatch.setattr(ops, name, lambda *a, **k: None)
    for rows, want in left_out.items():
        took.clear()
        ctx = SimpleNamespace(env=CTX.env, rows=rows, alloc=lambda shape, dtype=BF16: empty(*shape, dtype=dtype))
        part._routed(empty(rows, sizes["hidden"]), ctx, False)
        real, inter = sizes["real"], sizes["inter"]
        assert took == [want[0] and (real, 2 * inter, False), want[1] and (real, inter, True)], rows


@pytest.mark.parametrize("M,N,K,tile", [
    (2048, 3584, 18944, (128, 224)), (12001, 3584, 18944, (256, 224)),        # 256 tiles, 752: one round, three of the shorter ones
    (2048, 37888, 3584, (256, 256)), (203, 37888, 3584, (256, 160)), (100, 37888, 3584, (128, 160)),
    (2048, 4608, 3584, (128, 288)), (1, 4, 64, (128, 160))])
def test_which_tile_a_product_of_many_rows_takes(M, N, K, tile):
    assert ops.gemm_tall_tile(M, N, K) == tile


@pytest.mark.parametrize("N,K,tiles", [
    (37888, 3584, {70: (128, 160), 203: (256, 160), 300: (128, 224), 2048: (256, 256), 12001: (256, 256)}),
    (14336, 4096, {175: None, 512: (128, 224)}),        # 0.70 of a round; a whole one
    # whole rounds of two rows of tiles that are half padding: 1.1 to 1.24 of the time of the two launches
    (28672, 4096, {138: None, 203: (128, 224), 259: None, 345: None, 380: (256, 224)}),
    (37888, 2048, {70: (128, 160), 138: (256, 160), 541: None, 600: (256, 224), 784: None}),
    (9728, 896, {2048: None}), (37888, 3600, {2048: None}), (37884, 3584, {2048: None})])      # short K (tall_gated's), no multiples
def test_which_gated_products_of_longer_k_run_as_one_kernel(N, K, tiles):
    """At 256 units: where the tiles are 0.8 of their rounds or more, and one row of tiles or 0.72 of the rounds real outputs."""
    lin = Linear(empty(N, K))
    assert not any(lin.gated_tile(r, CTX, empty(r, K)) for r in tiles)      # no part has allowed it
    lin.one_round_tiles = True
    assert {r: lin.gated_tile(r, CTX, empty(r, K)) for r in tiles} == tiles
    with route_before_the_library(lambda c: c.N == N):
        assert not any(lin.gated_tile(r, CTX, empty(r, K)) for r in tiles)


@pytest.mark.parametrize("kind,names", [("gated_mlp", {"activation": "silu"}), ("dense_mlp", {"activation": "relu2"})])
def test_no_rows_are_no_product_in_tiles(monkeypatch, kind, names):
    """A part called with no rows answers with none, at a K and a width whose products of many rows run in tiles."""
    def alloc(shape, dtype=BF16):
        return empty(*shape, dtype=dtype)
    ctx = SimpleNamespace(env=CTX.env, rows=0, alloc=alloc, take_sink=lambda: None)
    part = build_part("feed_forward", PartSpec(kind, {"hidden_size": 2048, "intermediate_size": 16384, **names}), "m.", CTX.env)
    part.bind({k: empty(*v.shape) for k, v in part.tensor_specs().items()})
    for name in ("silu_mul", "unary_act"):
        monkeypatch.setattr(ops, name, lambda *a, **k: None)
    first = part.gate_up if kind == "gated_mlp" else part.up
    assert first.gated_tile(0, ctx, empty(0, 2048)) is None
    assert part.forward(empty(0, 2048), ctx).shape == (0, 2048)


@pytest.mark.parametrize("N,K,rows", [(3584, 18944, {768: False, 900: False, 1300: True, 1408: True, 2048: True, 2177: True, 3001: True, 12001: True}),
                                      # the library's tiles 0.88, 0.93, 0.98 and 1.97 of whole rounds; three rounds of 128 x 256
                                      (3584, 18944, {4096: True, 4229: False, 4608: False, 9120: False, 6889: False}),
                                      (5120, 27648, {900: True, 1180: True, 1537: True, 8192: True}), (4096, 14336, {1664: False, 10000: False}),
                                      (3584, 29568, {12001: False}), (8192, 29568, {768: False, 1024: False}), (2048, 8192, {4000: False}),
                                      (3584, 18912, {2048: False, 12001: False}), (3586, 18944, {2048: False, 12001: False})])
def test_which_products_of_long_k_run_in_tiles_of_many_rounds(N, K, rows):
    """At 256 units: K from 16448 to 27648, 0.7 of the rounds real outputs, the library's own tiles not all but whole rounds."""
    lin = Linear(empty(N, K))
    assert not any(lin._long(r, empty(r, K), empty(r, N), BF16) for r in rows)
    lin.one_round_tiles = True
    assert {r: lin._long(r, empty(r, K), empty(r, N), BF16) for r in rows} == rows
    assert not any(lin._long(r, empty(r, K), empty(r, N, dtype=torch.float32), torch.float32) for r in rows)


@pytest.mark.parametrize("M,N,K,taken", [
    (1003, 3584, 18944, True), (2048, 37888, 3584, True), (130, 37888, 3584, False),      # 126 of the second row of tiles are padding
    (700, 288, 32, False), (305, 3400, 64, True),                                         # one stage; two
    (532, 14083, 64, False), (946, 4567, 160, False), (1096, 989, 544, True),             # rows of results that are stored one by one
    (1003, 3584, 18948, False)])
def test_which_32_bit_products_run_in_whole_rounds(M, N, K, taken):
    """At 256 units, rows that begin at 16-byte boundaries."""
    from hector_engine_amd.kernels import lib
    assert lib.load().he_gemm_plain_in_rounds(M, N, K, int(N % 4 == 0)) == taken
