"""The rotation's launch writes v a row a workgroup up to 1,024 rows and eight rows a workgroup beyond: the same cache."""
import pytest
import torch

from hector_engine_amd.kernels import ops
from tests.test_kernels_gpu import PAGE, cached_v, dev, paged_setup, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [129, 1024, 1025])
def test_values_of_single_rows_and_runs_reach_their_places(rows):
    """Seven one-token sequences, then a run that begins inside a group of eight keys."""
    KVH, hd, H = 2, 64, 2
    lengths = [5, 64, 70, 8, 127, 1, 33, 13]
    new = [1] * 7 + [rows - 7]
    slots, table, kpool, vpool = paged_setup([a + b for a, b in zip(lengths, new)], KVH, hd, torch.bfloat16, 20)
    qkv = rnd(rows, (H + 2 * KVH) * hd, seed=21).bfloat16()
    positions = torch.cat([torch.arange(a, a + b) for a, b in zip(lengths, new)]).int()
    row_seq = torch.cat([torch.full((b,), i) for i, b in enumerate(new)]).int()
    kp, vp = dev(kpool), dev(vpool)
    ops.qkv_rope_cache(torch.zeros(rows, H * hd, dtype=torch.bfloat16, device="cuda"), kp, vp, dev(qkv), H * hd, KVH * hd, None,
                       dev(positions), dev(row_seq), dev(torch.tensor(slots, dtype=torch.int32)), dev(table), None, 0, rows, H,
                       KVH, hd, True)
    v = qkv[:, (H + KVH) * hd:].reshape(rows, KVH, hd)
    vp = vp.cpu()
    for r in range(rows):
        page = table[slots[row_seq[r]], positions[r] // PAGE].item()
        assert torch.equal(cached_v(vp, page, positions[r] % PAGE, hd), v[r])
    assert (vp != 0).sum() == (v != 0).sum()
