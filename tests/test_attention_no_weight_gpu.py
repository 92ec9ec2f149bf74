"""Keys whose score is -inf have no weight, however a page of them lies among others; scores that are no numbers stay visible; a
sink of -inf is no sink. All forms of the plain attention: 32-bit on the matrix cores (head size 64) and by the vector ALU
(80), bf16; many queries, one query over all pages, one query page by page."""
import math

import pytest
import torch

from hector_engine_amd.kernels import ops
from tests.test_kernels_gpu import dev, fill_cache, paged_setup, rnd

pytestmark = pytest.mark.gpu
H, KVH, N = 2, 1, 200


def setting(hd, dtype, seed=70):
    slots, table, kpool, vpool = paged_setup([N], KVH, hd, dtype, seed)
    k, v = rnd(N, KVH, hd, seed=seed + 1).to(dtype), rnd(N, KVH, hd, seed=seed + 2).to(dtype)
    fill_cache(table, slots, kpool, vpool, [k], [v])
    q = rnd(N, H, hd, seed=seed + 3).to(dtype)
    return (dev(kpool), dev(vpool), dev(torch.tensor(slots, dtype=torch.int32)), dev(table)), q, k, v


def run(fixed, q, lo, hi, split, **more):
    kpool, vpool, slot, table = fixed
    hd, ws = q.shape[-1], None
    out = torch.full((hi - lo, H * hd), 7.0, dtype=q.dtype, device="cuda")
    if split:
        ws = torch.empty(ops.attention_plain_workspace_floats(hi - lo, H, hd, N, 0, 0), device="cuda")
    ops.attention_plain(out, dev(q[lo:hi].reshape(hi - lo, -1)), kpool, vpool, dev(torch.arange(lo, hi).int()),
                        torch.zeros(hi - lo, dtype=torch.int32, device="cuda"), slot, table, hi - lo, H, KVH, hd, 0,
                        1.0 / math.sqrt(hd), N if split else 0, ws, **more)
    return out.view(hi - lo, H, hd)


def by_hand(q, k, v, lo, hi, bias, sinks):
    s = torch.einsum("qhd,kd->hqk", q[lo:hi].double(), k[:, 0].double()) / math.sqrt(q.shape[-1])
    gap = torch.arange(lo, hi)[:, None] - torch.arange(N)[None]
    s = s + bias.double()[:, gap.clamp(0, bias.shape[1] - 1)]
    s = s.masked_fill(gap < 0, -math.inf)
    top = s.amax(-1, keepdim=True).clamp(min=-1e30)
    w = torch.exp(s - top)
    total = w.sum(-1, keepdim=True) + (torch.exp(sinks.double()[:, None, None] - top) if sinks is not None else 0)
    return torch.einsum("hqk,kd->qhd", torch.where(w > 0, w / total, w), v[:, 0].double())


@pytest.mark.parametrize("hd,dtype", [(64, torch.float32), (80, torch.float32), (64, torch.bfloat16)])
@pytest.mark.parametrize("lo,hi,split", [(0, N, False), (150, 160, False), (150, 160, True)])
def test_keys_without_weight(hd, dtype, lo, hi, split):
    fixed, q, k, v = setting(hd, dtype)
    tol = 3e-6 if dtype == torch.float32 else 2 ** -7      # a few fp32 roundings of results of size 1; the rounding to bf16
    far, near, none = (torch.zeros(H, N) for _ in range(3))
    far[:, 20:] = -math.inf            # whole pages of earlier keys, and a page that begins with such keys
    near[:, :140] = -math.inf          # whole pages of later keys; the first 140 queries see no key at all
    near[1] = 0.0
    none[:] = -math.inf
    for bias in (far, near, none):
        for sinks in (None, torch.tensor([0.5, -math.inf])):
            got = run(fixed, q, lo, hi, split, table=dev(bias), sinks=None if sinks is None else dev(sinks))
            want = by_hand(q, k, v, lo, hi, bias, sinks)
            assert torch.allclose(got.cpu().double(), want, rtol=tol, atol=tol)


@pytest.mark.parametrize("hd,dtype", [(64, torch.float32), (80, torch.float32), (64, torch.bfloat16)])
@pytest.mark.parametrize("lo,hi,split", [(0, N, False), (150, 160, False), (150, 160, True)])
def test_scores_that_are_no_numbers_stay_visible(hd, dtype, lo, hi, split):
    fixed, q, k, v = setting(hd, dtype)
    bias = torch.zeros(H, N)
    bias[0, 100:164] = math.nan        # some page of a query at 164 and later, or a part of one
    got = run(fixed, q, lo, hi, split, table=dev(bias)).cpu()
    seen = max(0, 100 - lo)
    assert got[seen:, 0].isnan().all() and not got[:, 1].isnan().any() and not got[:seen].isnan().any()
