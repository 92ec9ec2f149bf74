"""Feed-forwards of many rows through the tile kernels, at sizes whose rules choose them: a part hands over the right rows,
weights and constants, turn by turn, and its results are those of 64-bit sums."""
from types import SimpleNamespace

import pytest
import torch

from hector_engine_amd.engine.scratch import ScratchPool
from hector_engine_amd.kernels import ops
from hector_engine_amd.parts.base import BuildEnv, PartSpec, build_part

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(BF16)


def bound_part(kind, params, scale):
    part = build_part("feed_forward", PartSpec(kind, params), "m.", BuildEnv(torch.device("cuda:0"), BF16, True))
    part.bind({k: rnd(*v.shape, seed=i, scale=scale) for i, (k, v) in enumerate(part.tensor_specs().items())})
    return part


def context(rows):
    scratch = ScratchPool(torch.device("cuda:0"))
    return SimpleNamespace(rows=rows, env=BuildEnv(torch.device("cuda:0"), BF16, True), scratch=scratch,
                           alloc=lambda shape, dtype=BF16: scratch.alloc(shape, dtype or BF16), take_sink=lambda: None, sink=None)


def spied(monkeypatch, name):
    """The calls of ops.<name>, each with its arguments and (for the first tensor) what it held afterwards."""
    calls, real = [], getattr(ops, name)

    def spy(*args, **kw):
        real(*args, **kw)
        calls.append(SimpleNamespace(args=[a.clone() if i in (0, 1) and isinstance(a, torch.Tensor) else a for i, a in enumerate(args)], kw=kw))
    monkeypatch.setattr(ops, name, spy)
    return calls


# A sum of K products in fp32 on the matrix cores: a chain of K / 32 additions and a tree of 32 in each, in units of
# 2^-24 of the sum of magnitudes (64-bit reference).
def sums(x, w):
    x, w = x.double(), w.double()
    K = x.shape[1]
    return x @ w.T, (K / 32 + 32) * 2 ** -24 * (x.abs() @ w.abs().T)


def gated(x, gate, up, fn, shift, limit):
    """The activation in 64 bits and how far a correct one may be off: gate and up carry the error of their sums and a rounding to bf16
    (8 bits: 2^-8 at most), the activation's derivative is at most 1.2 (|up| + shift) by gate and |gate| by up, the result is rounded to bf16."""
    g, eg = sums(x, gate)
    u, eu = sums(x, up)
    eg, eu = eg + 2 ** -8 * (g.abs() + eg), eu + 2 ** -8 * (u.abs() + eu)
    if limit:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    a = fn(g) * (u + shift)
    return a, 1.2 * (u.abs() + eu + shift) * eg + (g.abs() + eg) * eu + 1e-5 * a.abs()


SILU = (torch.nn.functional.silu, 0.0, 0.0)


@pytest.mark.parametrize("act,params,fn,shift,limit,consts", [
    ("silu", {}, *SILU, (1.0, 0.0, 0.0, 0.0)),
    ("gelu_tanh", {}, lambda g: torch.nn.functional.gelu(g, approximate="tanh"), 0.0, 0.0, (1.5957691216, 0.0, 0.0, 0.0713548162)),
    ("clamped_swiglu", {"limit": 1.5}, lambda g: g * torch.sigmoid(1.702 * g), 1.0, 1.5, (1.702, 1.5, 1.0, 0.0))])
@pytest.mark.parametrize("hidden,inter,turns", [(896, 4864, {600: 128}), (896, 4864, {1300: 256}), (256, 512, {8192: 128, 71: 0})])
def test_gated_products_as_one_kernel(monkeypatch, act, params, fn, shift, limit, consts, hidden, inter, turns):
    part = bound_part("gated_mlp", {"hidden_size": hidden, "intermediate_size": inter, "activation": act, **params}, hidden ** -0.5)
    rows = sum(turns)
    x, calls = rnd(rows, hidden, seed=90), spied(monkeypatch, "gemm_tall")
    out = part.forward(x, context(rows))
    assert [(c.args[4], c.kw["bm"]) for c in calls] == [t for t in turns.items() if t[1]]
    w = part.gate_up.weight
    for c in calls:
        assert c.kw["act"] == pytest.approx(consts)
        n = c.args[4]
        want, off = gated(x[:n], w[0::2], w[1::2], fn, shift, limit)
        assert ((c.args[0][:n].double() - want).abs() <= off + 2 ** -8 * (want.abs() + off)).all()
        down, err = sums(c.args[0][:n], part.down.weight)
        assert ((out[:n].double() - down).abs() <= err + 2 ** -8 * (down.abs() + err)).all()
    if len(turns) > 1:                                     # the last turn, which the library's product takes
        n = list(turns)[0]
        h, off = gated(x[n:], w[0::2], w[1::2], fn, shift, limit)
        off = off + 2 ** -8 * (h.abs() + off)
        down, err = sums(h, part.down.weight)
        err = err + off @ part.down.weight.double().abs().T
        assert ((out[n:].double() - down).abs() <= err + 2 ** -8 * (down.abs() + err)).all()


@pytest.mark.parametrize("rows,tall", [(7901, [7901]), (8192 + 71, [8192])])
def test_products_of_long_k_in_tiles(monkeypatch, rows, tall):
    part = bound_part("gated_mlp", {"hidden_size": 768, "intermediate_size": 16448}, 768 ** -0.5)
    x, calls = rnd(rows, 768, seed=91), spied(monkeypatch, "gemm_tall")
    out = part.forward(x, context(rows))
    assert [(c.args[4], c.kw["bm"], c.kw.get("act")) for c in calls] == [(n, 128, None) for n in tall]
    for c in calls:
        n = c.args[4]
        assert c.args[2] is part.down.weight and torch.equal(out[:n], c.args[0][:n])
        h, w = c.args[1][:n], part.gate_up.weight
        want, err = sums(h, part.down.weight)
        assert ((out[:n].double() - want).abs() <= err + 2 ** -8 * (want.abs() + err)).all()
        del want, err
        some = slice(n - 200, n)
        want, off = gated(x[some], w[0::2], w[1::2], *SILU)
        assert ((h[some].double() - want).abs() <= off + 2 ** -8 * (want.abs() + off)).all()
    if rows > tall[0]:
        w = part.gate_up.weight
        h, off = gated(x[tall[0]:], w[0::2], w[1::2], *SILU)
        off = off + 2 ** -8 * (h.abs() + off)
        want, err = sums(h, part.down.weight)
        err = err + off @ part.down.weight.double().abs().T
        assert ((out[tall[0]:].double() - want).abs() <= err + 2 ** -8 * (want.abs() + err)).all()


D = 1024
MLP = {"hidden_size": D, "intermediate_size": 192}


@pytest.mark.parametrize("turns", [(65,), (300,), (4096, 70), (4096, 9)])
@pytest.mark.parametrize("form", ["plain", "identity_limited", "beside_a_shared_expert"])
def test_experts_over_the_rows_that_chose_them(monkeypatch, form, turns):
    rows, real, top, I = sum(turns), 64, 4, 512
    more = {"plain": {}, "identity_limited": {"identity_experts": 3, "limit": 1.5},
            "beside_a_shared_expert": {"shared": {"gate": "sg", "feed_forward": PartSpec("gated_mlp", MLP)}}}[form]
    part = bound_part("routed_experts", {"hidden_size": D, "intermediate_size": I, "experts": real, "top": top,
                                         "correction": False, **more}, D ** -0.5)
    name, n_at = ("routed_groups_act", 6) if form == "beside_a_shared_expert" else ("routed_groups", 10)
    x, calls, ctx = rnd(rows, D, seed=92), spied(monkeypatch, name), context(rows)
    routed = part._routed(x, ctx, False)
    assert [c.args[n_at] for c in calls] == list(turns)
    assert {c.kw["bm"] for c in calls} == {part._many_rows(rows, x, ctx)} == {256 if rows > 4096 else 128}
    dense, ids = torch.empty(rows, real + 1, device="cuda"), torch.empty(rows, top, dtype=torch.int32, device="cuda")
    ops.route_tokens(dense, ids, torch.empty(rows, top, device="cuda"), None, None, rows, real, 1, 1, top, part.scale, x=x,
                     router=part.router)
    fn, shift, limit = (lambda g: g * torch.sigmoid(1.702 * g), 1.0, 1.5) if "limit" in more else SILU
    want = torch.zeros(rows, D, dtype=torch.float64, device="cuda")
    err = torch.zeros_like(want)
    wide = torch.zeros(rows, real * I, dtype=torch.float64, device="cuda")
    wide_off = torch.zeros_like(wide)
    for e in range(real):
        w, cols = part.gate_up.weight[2 * e * I:2 * (e + 1) * I], slice(e * I, (e + 1) * I)
        a, off = gated(x, w[0::2], w[1::2], fn, shift, limit)
        f = dense[:, e:e + 1].double()
        wide[:, cols], wide_off[:, cols] = a * f, (off + 2 ** -8 * (a.abs() + off)) * f
        d = part.down.weight[:, cols].double()
        want += wide[:, cols] @ d.T
        err += wide_off[:, cols] @ d.abs().T
    err += (real * I / 32 + 32) * 2 ** -24 * (wide.abs() @ part.down.weight[:, :real * I].double().abs().T)
    if "identity_experts" in more:
        assert (ids >= real).any()
        want += dense[:, real:].double() * x.double()
        err += 2 ** -22 * (dense[:, real:].double() * x.double()).abs()
    assert ((routed.double() - want).abs() <= err + 2 ** -8 * (want.abs() + err)).all()
    if form == "beside_a_shared_expert":
        got = torch.cat([c.args[0][:n] for c, n in zip(calls, turns)]).double()
        assert ((got - wide).abs() <= wide_off).all()                    # exact zeros where an expert was not chosen
        both = torch.empty(rows, D, dtype=BF16, device="cuda")
        ops.gated_add(both, routed, part.shared.forward(x, context(rows)), x, part.shared_gate, rows)
        assert torch.equal(part.forward(x, context(rows)), both)


@pytest.mark.parametrize("form", [{}, {"identity_experts": 2}, {"shared": {"feed_forward": PartSpec("gated_mlp", {"hidden_size": 1024, "intermediate_size": 1088})}}])
@pytest.mark.parametrize("rows", [3, 5])
def test_experts_that_nobody_chose_are_left_out(monkeypatch, form, rows):
    """A step of few rows at sizes whose rule leaves them out of both products: the bits of the products over all experts."""
    part = bound_part("routed_experts", {"hidden_size": 1024, "intermediate_size": 1088, "experts": 64, "top": 12, "correction": False, **form},
                      1024 ** -0.5)
    x = rnd(rows, 1024, seed=94)
    assert part._leaves_out(rows) == (True, True) and not part._few_rows(rows, x, context(rows))
    out = part._routed(x, context(rows), False)
    monkeypatch.setattr(part, "_leaves_out", lambda rows: (False, False))
    assert torch.equal(out, part._routed(x, context(rows), False))


@pytest.mark.parametrize("act,params,fn,shift,limit,consts", [
    ("silu", {}, *SILU, (1.0, 0.0, 0.0, 0.0)),
    ("clamped_swiglu", {"limit": 1.5}, lambda g: g * torch.sigmoid(1.702 * g), 1.0, 1.5, (1.702, 1.5, 1.0, 0.0))])
@pytest.mark.parametrize("inter,rows,tile", [(20000, 70, (128, 160)), (12200, 250, (128, 224)), (2872, 1900, (256, 192))])
def test_gated_products_of_longer_k_as_one_kernel(monkeypatch, act, params, fn, shift, limit, consts, inter, rows, tile):
    """K of 1088, above the rule for short ones; columns and rows that end inside a tile."""
    hidden = 1088
    part = bound_part("gated_mlp", {"hidden_size": hidden, "intermediate_size": inter, "activation": act, **params}, hidden ** -0.5)
    x, calls = rnd(rows, hidden, seed=92), spied(monkeypatch, "gemm_tall")
    part.forward(x, context(rows))
    assert [(c.args[4], (c.kw["bm"], c.kw["bn"])) for c in calls] == [(rows, tile)]
    assert calls[0].kw["act"] == pytest.approx(consts)
    w = part.gate_up.weight
    want, off = gated(x, w[0::2], w[1::2], fn, shift, limit)
    assert ((calls[0].args[0][:rows].double() - want).abs() <= off + 2 ** -8 * (want.abs() + off)).all()


@pytest.mark.parametrize("rows,kernel", [(1, "gemm_blocksplit"), (5, "gemm_blocksplit"), (16, "gemm_blocksplit"), (17, None), (70, "gemm_tall"), (1900, "gemm_tall")])
@pytest.mark.parametrize("kind", ["relu2", "relu", "gelu_tanh", "silu"])
def test_activations_that_go_with_the_up_product(monkeypatch, rows, kernel, kind):
    """The bits of the product and the activation one after the other; the relu ones also in steps of many rows."""
    hidden, inter = 1088, 40000 if rows == 70 else 5744
    part = bound_part("dense_mlp", {"hidden_size": hidden, "intermediate_size": inter, "activation": kind}, hidden ** -0.5)
    x, w = rnd(rows, hidden, seed=93), part.up.weight
    alone = torch.empty(rows, inter, dtype=BF16, device="cuda")
    if rows <= 16:
        ops.gemm_blocksplit(alone, x, w, None, rows)
    elif kernel:
        ops.gemm_tall(alone, x, w, None, rows)
    if kernel:
        ops.unary_act(alone, alone, rows, kind)
    one, two = spied(monkeypatch, kernel or "gemm_tall"), spied(monkeypatch, "unary_act")
    h = part._activated(x, rows, context(rows))
    taken = kernel and (rows <= 16 or kind.startswith("relu"))
    assert [c.kw.get("unary") for c in one] == ([kind] if taken or rows <= 16 else []) and len(two) == (0 if taken else 1)
    if taken:
        assert torch.equal(h[:rows], alone)
