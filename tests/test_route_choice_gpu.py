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
