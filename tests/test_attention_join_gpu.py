"""One-token attention whose keys are cut across workgroups: the parts joined by the workgroup that finishes last give the bits of
the join by a second launch."""
import math

import pytest
import torch

from tests.plain import qwen2_plain as P
from tests.test_kernels_gpu import dev, fill_cache, from_pieces, ops, paged_setup, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KVH,hd", [(14, 2, 64), (28, 4, 128), (40, 2, 128), (3, 3, 64)])
@pytest.mark.parametrize("lengths,max_keys,spread", [([530], 1024, False), ([700, 1, 2050], 4096, False), ([3000] + [40] * 30, 20000, True),
                                                     ([1], 256, False), ([2500], 20000, False)])
def test_the_last_workgroup_joins_with_the_same_bits(ops, H, KVH, hd, lengths, max_keys, spread):
    """One to 32 parts, parts without keys, tiles of 16 heads of a group (20 heads a kv head), a padding row, both layouts of the
    result. Every launch finds another workspace (NaN) and leaves the counters as it found them."""
    B, rows = len(lengths), len(lengths) + 1
    slots, table, kpool, vpool = paged_setup(lengths, KVH, hd, torch.bfloat16, 60)
    fill_cache(table, slots, kpool, vpool, [rnd(n, KVH, hd, seed=61 + i).bfloat16() for i, n in enumerate(lengths)],
               [rnd(n, KVH, hd, seed=171 + i).bfloat16() for i, n in enumerate(lengths)])
    qkv = dev(rnd(rows, (H + 2 * KVH) * hd, seed=81, scale=1.5).bfloat16())
    bias, inv, table = dev(rnd((H + 2 * KVH) * hd, seed=82).bfloat16()), dev(P.rope_inv_freq(hd, 50000.0)), dev(table)
    i32 = lambda v: dev(torch.tensor(v, dtype=torch.int32))
    positions, row_seq, seq_slot = i32([0] + [n - 1 for n in lengths]), i32([-1] + list(range(B))), i32(slots)
    floats = ops.attention_decode_fused_workspace_floats(rows, H, KVH, hd, max_keys, spread)
    groups = rows * KVH * -(-H // KVH // 16)
    counters = torch.zeros(groups, dtype=torch.int32, device="cuda")

    def run(pieces, counters):
        out = torch.full(ops.pieces_shape(rows, H * hd) if pieces else (rows, H * hd), float("nan"), dtype=torch.bfloat16, device="cuda")
        kp, vp = dev(kpool), dev(vpool)
        ws = torch.full((floats,), float("nan"), device="cuda") if floats else None
        ops.attention_decode_fused(out, qkv, bias, kp, vp, positions, row_seq, seq_slot, table, inv, hd, rows, H, KVH, hd, 0,
                                   1.0 / math.sqrt(hd), max_keys, True, ws, out_pieces=pieces, spread=spread, counters=counters)
        return (from_pieces(out) if pieces else out).cpu()

    want = run(False, None)
    assert want[0].abs().max() == 0 and bool(torch.isfinite(want).all())
    for again in range(3):
        assert torch.equal(run(False, counters), want)
        assert torch.equal(run(True, counters), want)
        assert not counters.any()
    if groups > 1:
        few = torch.full((groups - 1,), 77, dtype=torch.int32, device="cuda")      # too few: not used
        assert torch.equal(run(False, few), want) and bool((few == 77).all())


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("G", [17, 20, 33])
def test_tiles_of_heads_give_the_bits_of_groups_of_their_own(ops, hd, G):
    """A group of more than 16 query heads, whose tiles walk the same keys by way of the caches, beside groups of 16 heads and fewer, whose keys are read
    past them: in one launch and in two, 1 to 250 keys."""
    KVH, lengths, max_keys = 2, [1, 33, 64, 250], 256
    B, H = len(lengths), 2 * G
    slots, table, kpool, vpool = paged_setup(lengths, KVH, hd, torch.bfloat16, 40)
    fill_cache(table, slots, kpool, vpool, [rnd(n, KVH, hd, seed=61 + i).bfloat16() for i, n in enumerate(lengths)],
               [rnd(n, KVH, hd, seed=171 + i).bfloat16() for i, n in enumerate(lengths)])
    qkv = dev(rnd(B, (H + 2 * KVH) * hd, seed=81, scale=1.5).bfloat16())
    inv, table = dev(P.rope_inv_freq(hd, 50000.0)), dev(table)
    i32 = lambda v: dev(torch.tensor(v, dtype=torch.int32))
    positions, row_seq, seq_slot = i32([n - 1 for n in lengths]), i32(range(B)), i32(slots)

    def run(first, count, fused):
        """The heads first .. first + count of both groups as groups of their own."""
        q = qkv[:, :H * hd].view(B, KVH, G, hd)[:, :, first:first + count].reshape(B, -1)
        if fused:
            out = torch.empty(B, KVH * count * hd, dtype=torch.bfloat16, device="cuda")
            floats = ops.attention_decode_fused_workspace_floats(B, KVH * count, KVH, hd, max_keys, False)
            assert floats == 0
            ops.attention_decode_fused(out, torch.cat([q, qkv[:, H * hd:]], 1).contiguous(), None, dev(kpool), dev(vpool), positions, row_seq, seq_slot, table,
                                       inv, hd, B, KVH * count, KVH, hd, 0, hd ** -0.5, max_keys, True, None)
        else:
            out = torch.empty(B, KVH * count, hd, dtype=torch.bfloat16, device="cuda")
            ws = torch.empty(ops.attention_decode_workspace_floats(B, KVH * count, KVH, hd, max_keys), device="cuda")
            ops.attention_decode(out, q.reshape(B, -1, hd).contiguous(), dev(kpool), dev(vpool), positions, row_seq, seq_slot, table, B, KVH * count, KVH, hd, 0,
                                 hd ** -0.5, max_keys, ws)
        return out.view(B, KVH, count, hd)
    for fused in (True, False):
        whole = run(0, G, fused)
        assert bool(torch.isfinite(whole.float()).all()) and whole.abs().max() > 0
        for first in range(0, G, 16):
            assert torch.equal(whole[:, :, first:first + 16], run(first, min(16, G - first), fused))
