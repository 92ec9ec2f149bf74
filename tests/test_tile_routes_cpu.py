"""Which products of many rows run through the tile kernels: the rules alone, over tensors without storage."""
import contextlib
from types import SimpleNamespace

import pytest
import torch

from hector_engine_amd.kernels import routes
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
