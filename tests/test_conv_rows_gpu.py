"""The convolution of a step with work for the whole chip: eight rows and four channels a thread give the bits of a row and channel a thread."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,C", [(2, 4096), (3, 5124), (4, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_runs_of_rows(K, C, dtype):
    """Sequences that begin anywhere in a block of eight rows, of one row up, with and without rows before the step, padding rows, a view of
    wider rows; the same sequences one after the other in steps too small for the kernel give the same rows and the same carried inputs."""
    from hector_engine_amd.kernels import ops
    lengths = [700, 1, 2, 3, 9, 130, 5, 170]
    rows, pad = sum(lengths), 30
    assert (rows + pad) * C >= 1 << 22 > max(lengths) * C
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(rows + pad, C + 8, generator=g, device="cuda").to(dtype)[:, 4:4 + C]
    taps, bias = torch.randn(C, K, generator=g, device="cuda").bfloat16(), torch.randn(C, generator=g, device="cuda").bfloat16()
    state = torch.randn(len(lengths), (K - 1) * C + 4, generator=g, device="cuda").view(torch.uint8).view(len(lengths), -1)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    starts = [11 * (i % 3) for i in range(len(lengths))]
    cu = [0] + torch.tensor(lengths).cumsum(0).tolist()

    def run(which, x, pad):
        """The sequences `which`, whose rows are x, in one step."""
        lens = [lengths[i] for i in which]
        pos = sum((list(range(starts[i], starts[i] + lengths[i])) for i in which), []) + [0] * pad
        seq = sum(([k] * n for k, n in enumerate(lens)), []) + [-1] * pad
        out = torch.full((len(x), C), 7.0, dtype=dtype, device="cuda")
        ops.conv_state(out, x, taps, bias, carried, i32(pos), i32(seq), i32([len(lengths) - 1 - i for i in which]), i32([starts[i] for i in which]),
                       i32([0] + torch.tensor(lens).cumsum(0).tolist()), len(x), len(which), False)
        return out

    carried = state.clone()
    got, after = run(range(len(lengths)), x, pad), carried
    carried = state.clone()
    want = torch.cat([run([i], x[cu[i]:cu[i + 1]], 0) for i in range(len(lengths))])
    assert torch.equal(got[:rows], want) and not got[rows:].any()
    assert torch.equal(after, carried)
