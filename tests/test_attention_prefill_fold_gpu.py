"""Prompt attention in parts where the heads of a kv group share a workgroup's 128 columns: sequences of up to 128 / G new
tokens beside longer ones."""
import pytest
import torch

from tests.test_kernels_gpu import attention_case, dev, ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KVH,hd,window", [(14, 2, 128, 0), (8, 2, 64, 0), (8, 2, 64, 100), (3, 3, 80, 0), (40, 1, 16, 300)])
@pytest.mark.parametrize("parts", [2, 7, 32])
def test_folded_beside_longer_sequences(ops, H, KVH, hd, window, parts):
    """Per group size G: one token, the most that share a workgroup (128 // G), one more than that, a longest one of two blocks, and
    a one-token sequence of one key (parts without pages). Tolerance as the kernel's other tests: bf16 operands and results."""
    most = 128 // (H // KVH)
    q_lens = [1, most, most + 1, 200, 1, min(2, most)]
    lengths = [900, 700 + most, 64 * 9 + most + 1, 1000, 1, 65]
    got, want = attention_case(ops, "prefill", torch.bfloat16, H, KVH, hd, window, lengths, q_lens, 61, tiles=2, parts=parts)
    for g, w in zip(got, want):
        assert torch.allclose(g, w, rtol=2 ** -6, atol=2 ** -6)


def test_many_sequences_are_counted_in_turns_of_64(ops):
    """130 sequences, short and long ones mixed: the search goes through three turns of 64 of them."""
    q_lens = [(1, 2, 150, 40)[i % 4] for i in range(130)]
    lengths = [m + 37 * (i % 11) for i, m in enumerate(q_lens)]
    got, want = attention_case(ops, "prefill", torch.bfloat16, 4, 1, 64, 0, lengths, q_lens, 62, tiles=2, parts=2)
    for g, w in zip(got, want):
        assert torch.allclose(g, w, rtol=2 ** -6, atol=2 ** -6)


def test_rows_of_no_sequence_get_zeros(ops):
    """The join of parts writes zeros into the rows behind the last sequence's, whatever workspace and result held."""
    H, KVH, hd, rows, pad, parts = 4, 2, 64, 20, 13, 3
    q = torch.randn(rows + pad, H * hd, generator=torch.Generator().manual_seed(1)).bfloat16()
    pool = torch.zeros(8, KVH, 64 * hd, dtype=torch.bfloat16, device="cuda")
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    out = torch.full((rows + pad, H * hd), float("nan"), dtype=torch.bfloat16, device="cuda")
    ws = torch.full((ops.attention_prefill_workspace_floats(rows + pad, H, hd, parts),), float("nan"), device="cuda")
    ops.attention_prefill(out, dev(q), pool, pool, i32(0, rows, rows, rows), i32(0, -1, -1), i32(300, 0, 0),
                          torch.arange(8, dtype=torch.int32, device="cuda").reshape(1, 8), 3, 32, rows + pad, H, KVH, hd, 0,
                          0.125, kernel=2, parts=parts, workspace=ws)
    assert torch.equal(out.cpu().float(), torch.zeros(rows + pad, H * hd))     # values of zero, and zeros


def test_parts_of_steps_whose_other_sequences_are_short(ops):
    """The rule with the step's rows and kv heads: the other sequences share what the longest leaves."""
    assert ops.attention_prefill_parts(8, 256, 28, 128, 4096, 256, 4) == 6       # 512 // (2 * 28 + 7 * 4)
    assert ops.attention_prefill_parts(8, 256, 28, 128, 4096) == 1               # eight sequences of 256
    assert ops.attention_prefill_parts(8, 256, 28, 128, 1000, 256, 4) == 1       # fewer than four keys a query
    assert ops.attention_prefill_parts(1, 8, 28, 128, 8064, 8, 4) == 31          # one folded sequence: four pages a part
    assert ops.attention_prefill_parts(4, 128, 28, 128, 4096, 512, 4) == ops.attention_prefill_parts(4, 128, 28, 128, 4096) == 4
    # one sequence and padding rows behind it
    assert ops.attention_prefill_parts(1, 200, 28, 128, 8200, 256, 4) == ops.attention_prefill_parts(1, 200, 28, 128, 8200) == 9
