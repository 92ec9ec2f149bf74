"""The 32-bit attention on the matrix cores (head sizes 32, 64, 96, 128): its three launches (runs of queries, one query over all
pages, one query page by page) give the same bits, and a value that is not finite reaches only the queries that see it."""
import math

import pytest
import torch

from hector_engine_amd.kernels import ops
from tests.plain import qwen2_plain as P
from tests.test_kernels_gpu import dev, fill_cache, paged_setup, rnd

pytestmark = pytest.mark.gpu
F32 = torch.float32


class Step:
    """Sequences of `lengths` keys of which the last `q_lens` positions are queries."""

    def __init__(self, H, KVH, hd, lengths, q_lens, seed, spoil=None):
        self.H, self.KVH, self.hd, self.lengths, self.q_lens = H, KVH, hd, lengths, q_lens
        slots, table, kpool, vpool = paged_setup(lengths, KVH, hd, F32, seed)
        self.ks = [rnd(n, KVH, hd, seed=seed + 1 + i) for i, n in enumerate(lengths)]
        self.vs = [rnd(n, KVH, hd, seed=seed + 50 + i) for i, n in enumerate(lengths)]
        if spoil is not None:
            spoil(self)
        fill_cache(table, slots, kpool, vpool, self.ks, self.vs)
        self.qs = [rnd(m, H, hd, seed=seed + 100 + i, scale=2.0) for i, m in enumerate(q_lens)]
        self.q = dev(torch.cat(self.qs).reshape(-1, H * hd))
        self.positions = dev(torch.cat([torch.arange(n - m, n) for n, m in zip(lengths, q_lens)]).int())
        self.row_seq = dev(torch.cat([torch.full((m,), i) for i, m in enumerate(q_lens)]).int())
        self.fixed = (dev(kpool), dev(vpool)), (dev(torch.tensor(slots, dtype=torch.int32)), dev(table))

    def run(self, lo, hi, window=0, split=False, **more):
        (kpool, vpool), (slot, table) = self.fixed
        out = torch.full((hi - lo, self.H * self.hd), 7.0, device="cuda")
        more = {k: (v[lo:hi] if k == "gate" else v) for k, v in more.items()}
        most, ws = 0, None
        if split:
            most = max(self.lengths)
            floats = ops.attention_plain_workspace_floats(hi - lo, self.H, self.hd, most, window, more.get("chunk", 0))
            assert floats > 0
            ws = torch.empty(floats, device="cuda")
        ops.attention_plain(out, self.q[lo:hi].contiguous(), kpool, vpool, self.positions[lo:hi].contiguous(),
                            self.row_seq[lo:hi].contiguous(), slot, table, hi - lo, self.H, self.KVH, self.hd, window,
                            1.0 / math.sqrt(self.hd), most, ws, **more)
        return out


@pytest.mark.parametrize("H,KVH,hd", [(28, 4, 128), (6, 3, 32), (4, 4, 96), (14, 2, 64), (40, 2, 64)])
@pytest.mark.parametrize("window,chunk,extras", [(0, 0, False), (70, 0, False), (0, 48, True), (0, 0, True)])
def test_runs_single_queries_and_pages_give_the_same_bits(H, KVH, hd, window, chunk, extras):
    # long runs, runs that end inside a group of 32 rows, runs of fewer than 8 rows, single tokens behind many keys
    step = Step(H, KVH, hd, [150, 333, 67, 1, 90, 200, 64], [150, 70, 9, 1, 3, 1, 40], 300)
    rows = sum(step.q_lens)
    more = {}
    if extras:
        more = dict(sinks=dev(rnd(H, seed=9)), gate=dev(rnd(rows, H, seed=10)), slopes=dev(rnd(H, seed=11).abs()))
    whole = step.run(0, rows, window, chunk=chunk, **more)
    for lo in range(0, rows, 29):
        hi = min(rows, lo + 29)
        assert torch.equal(step.run(lo, hi, window, chunk=chunk, **more), whole[lo:hi])
        if not chunk and not (window and hi - lo < 2):
            assert torch.equal(step.run(lo, hi, window, split=True, chunk=chunk, **more), whole[lo:hi])
    if not more and not chunk:
        r = 0
        for i, (n, m) in enumerate(zip(step.lengths, step.q_lens)):
            want = P.attention(step.qs[i].double(), step.ks[i].double(), step.vs[i].double(), torch.arange(n - m, n), torch.arange(n), window)
            assert torch.allclose(whole.cpu()[r:r + m].double().reshape(want.shape), want, rtol=3e-6, atol=3e-6)
            r += m


@pytest.mark.parametrize("what", [float("inf"), float("nan")])
def test_a_value_that_is_not_finite_reaches_only_the_queries_that_see_it(what):
    def spoil(step):
        step.vs[0][75, 1, 3] = what
    bad, good = (Step(4, 2, 64, [100], [100], 500, s) for s in (spoil, None))
    for lo, hi, split in ((0, 100, False), (60, 100, False), (70, 80, True)):
        got, want = bad.run(lo, hi, split=split).view(hi - lo, 4, 64), good.run(lo, hi, split=split).view(hi - lo, 4, 64)
        seen = max(0, 75 - lo)
        assert torch.equal(got[:seen], want[:seen]) and torch.equal(got[:, :2], want[:, :2])
        assert not got[seen:, 2:, 3].isfinite().any()
        keep = torch.arange(64) != 3
        assert torch.equal(got[:, :, keep.cuda()], want[:, :, keep.cuda()])


@pytest.mark.parametrize("hd,window", [(128, 0), (128, 300), (64, 0), (32, 0)])
def test_a_wavefront_takes_several_pages_of_a_query(hd, window):
    """32 queries of 8 heads of their own, of 1 to 16 pages, in more units than the chip holds at once when each is a page."""
    lengths = [1 + 33 * i for i in range(31)] + [1000]
    step = Step(16, 16, hd, lengths, [1] * 32, 700)
    split = step.run(0, 32, window, split=True)
    assert torch.equal(split, step.run(0, 32, window)) and torch.equal(split[31:], step.run(31, 32, window, split=True))
