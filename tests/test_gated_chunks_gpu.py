"""The matrix memory and the state-space scan by chunks of rows: against the recurrences in 64 bits and beside the walk row by
row, over edges of chunks, of blocks of key and value dims, and gates from keeping everything to forgetting at once."""
import pytest
import torch

pytestmark = pytest.mark.gpu
F64 = torch.float64


@pytest.fixture(scope="module")
def ops():
    from hector_engine_amd.kernels import ops
    return ops


def rnd(*shape, seed, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed), dtype=F64) * scale


def i32(*v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def cu_of(lengths):
    return i32(0, *torch.tensor(lengths).cumsum(0).tolist())


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


# first a step of these lengths, then one of those that goes on from its states (both have a sequence of more than 64 rows)
STEPS = [[130, 1, 64, 260, 65], [3, 200, 128, 1, 97]]


def mlstm_plain(q, k, v, i, f, state):
    """One head: q, k [T, dk], v [T, dv], logarithms i, f [T]; state (S, n, m) or None."""
    S, n, m = state or (torch.zeros(q.shape[1], v.shape[1], dtype=F64), torch.zeros(q.shape[1], dtype=F64), torch.zeros((), dtype=F64))
    y = []
    for t in range(len(q)):
        new = torch.maximum(f[t] + m, i[t])
        a, b = torch.exp(f[t] + m - new), torch.exp(i[t] - new)
        S, n, m = a * S + b * torch.outer(k[t], v[t]), a * n + b * k[t], new
        y.append(S.t() @ q[t] / (torch.maximum((n @ q[t]).abs(), torch.exp(-m)) + 1e-6))
    return torch.stack(y), (S, n, m)


@pytest.mark.parametrize("H,dk,dv", [(2, 128, 256), (3, 20, 36), (1, 8, 4), (2, 132, 68)])
@pytest.mark.parametrize("keep,write", [(3.0, -1.0), (-20.0, 0.0), (30.0, 12.0)])
def test_matrix_memory_by_chunks(ops, H, dk, dv, keep, write):
    slots, room = i32(2, 0, 4, 1, 3), 5
    state = {way: torch.zeros((room, 4 * ops.mlstm_state_floats(H, dk, dv)), dtype=torch.uint8, device="cuda") for way in ("chunks", "walk")}
    plain = [[None] * H for _ in range(5)]
    for s, lengths in enumerate(STEPS):
        rows = sum(lengths)
        x = rnd(rows, H * (2 * dk + dv), seed=s)
        if write > 1:                        # (every row is remembered: with signs of their own n . q would be a small difference)
            x[:, :2 * H * dk] = x[:, :2 * H * dk].abs()
        x = x.bfloat16()
        gates = torch.cat([rnd(rows, H, seed=10 + s, scale=2.0) + write, -torch.nn.functional.softplus(-(rnd(rows, H, seed=20 + s, scale=2.0) + keep))], 1).float()
        xd, gd, cu = x.cuda(), gates.cuda(), cu_of(lengths)
        q, k, v = xd[:, :H * dk], xd[:, H * dk:2 * H * dk], xd[:, 2 * H * dk:]
        floats = ops.mlstm_workspace_floats(rows, 5, max(lengths), H, dk, dv, torch.bfloat16)
        assert floats > 0
        got = {}
        for way in state:
            got[way] = torch.full((rows, H * dv), float("nan"), device="cuda")
            ws = torch.full((floats,), float("nan"), device="cuda") if way == "chunks" else None
            ops.mlstm_scan(got[way], q, k, v, gd, state[way], 0, cu, slots, rows, 5, H, dk, dv, dk ** -0.5, max_q_len=max(lengths), workspace=ws)
        want, r = torch.empty(rows, H * dv, dtype=F64), 0
        xq, g64 = x.double(), gates.double()
        for b, n in enumerate(lengths):
            at = slice(r, r + n)
            for h in range(H):
                cols = slice(h * dk, (h + 1) * dk)
                want[at, h * dv:(h + 1) * dv], plain[b][h] = mlstm_plain(
                    xq[at, :H * dk][:, cols] * dk ** -0.5, xq[at, H * dk:2 * H * dk][:, cols], xq[at, 2 * H * dk + h * dv:2 * H * dk + (h + 1) * dv],
                    g64[at, h], g64[at, H + h], plain[b][h])
            r += n
        e = {way: rel(got[way].cpu(), want) for way in got}
        # 32-bit sums and exponentials: a few 2^-24, the two about as far from 64 bits as each other (single inputs: a third either way)
        assert e["chunks"] <= 1.3 * e["walk"] < 1e-5


@pytest.mark.parametrize("rows,keep,positive", [(500, 0.0, False), (500, 3.0, True), (2048, 0.0, False)])
def test_matrix_memory_is_no_further_from_64_bits_than_the_walk(ops, rows, keep, positive):
    """Wide keys, whose sums are the longest, with memories that fade soon, and with products of one sign, whose sums' rounding does not
    average out: both are rounding errors of a few 2^-24, the chunks' no larger."""
    H, dk, dv = 4, 512, 256
    x = rnd(rows, H * (2 * dk + dv), seed=1)
    if positive:
        x[:, :2 * H * dk] = x[:, :2 * H * dk].abs()
    x = x.bfloat16().cuda()
    gates = torch.cat([rnd(rows, H, seed=2), -torch.nn.functional.softplus(-(rnd(rows, H, seed=3) + keep))], 1).float().cuda()
    q, k, v = x[:, :H * dk], x[:, H * dk:2 * H * dk], x[:, 2 * H * dk:]
    e = {}
    x64 = x.double()
    plain = [torch.zeros(*shape, dtype=F64, device="cuda") for shape in ((H, dk, dv), (H, dk), (H,))]
    want = mlstm_plain_heads(x64[:, :H * dk].reshape(rows, H, dk) * dk ** -0.5, x64[:, H * dk:2 * H * dk].reshape(rows, H, dk),
                             x64[:, 2 * H * dk:].reshape(rows, H, dv), gates[:, :H].double(), gates[:, H:].double(), plain).reshape(rows, H * dv)
    for way in ("chunks", "walk"):
        y, state = torch.empty(rows, H * dv, device="cuda"), torch.zeros((1, 4 * ops.mlstm_state_floats(H, dk, dv)), dtype=torch.uint8, device="cuda")
        ws = torch.empty(ops.mlstm_workspace_floats(rows, 1, rows, H, dk, dv, torch.bfloat16), device="cuda") if way == "chunks" else None
        ops.mlstm_scan(y, q, k, v, gates, state, 0, i32(0, rows), i32(0), rows, 1, H, dk, dv, dk ** -0.5, max_q_len=rows, workspace=ws)
        e[way] = rel(y, want)
    assert e["chunks"] <= e["walk"] < 1e-5


def test_matrix_memory_of_closed_gates(ops):
    """Input gates closed (-inf) for the first chunk and a half, then here and there; rows that forget everything (-inf) on either side of a
    chunk's edge: finite, and as the walk has it."""
    H, dk, dv, rows = 2, 32, 64, 200
    x = rnd(rows, H * (2 * dk + dv), seed=7).bfloat16().cuda()
    gates = torch.cat([rnd(rows, H, seed=8), -rnd(rows, H, seed=9).abs()], 1)
    gates[:96, 0] = -torch.inf
    gates[100:110, 1] = -torch.inf
    gates[[127, 128, 150], H] = -torch.inf
    gates[[20, 64], H + 1] = -torch.inf
    got = []
    for ws in (None, torch.full((ops.mlstm_workspace_floats(rows, 1, rows, H, dk, dv, torch.bfloat16),), float("nan"), device="cuda")):
        y = torch.empty(rows, H * dv, device="cuda")
        state = torch.zeros((1, 4 * ops.mlstm_state_floats(H, dk, dv)), dtype=torch.uint8, device="cuda")
        for at in (slice(0, 130), slice(130, rows)):
            n = at.stop - at.start
            ops.mlstm_scan(y[at], x[at, :H * dk], x[at, H * dk:2 * H * dk], x[at, 2 * H * dk:], gates[at].float().cuda(), state, 0, i32(0, n), i32(0), n, 1,
                           H, dk, dv, dk ** -0.5, max_q_len=n, workspace=ws)
        got.append(y.cpu().double())
    assert bool(torch.isfinite(got[0]).all()) and bool(torch.isfinite(got[1]).all())
    # both are fp32 sums; rows whose n . q is a small difference carry a few 2^-24 of what it is a difference of
    assert rel(got[1], got[0]) < 1e-4


@pytest.mark.parametrize("which", ["mlstm", "ssm"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_rows_before_one_that_is_not_finite(ops, which, bad):
    """A value that is no number, in the middle of a chunk: the rows before it are what they are without it, those behind it are no numbers
    in its column, as the walk has them, and the other columns never see it."""
    rows, at, col, bf16 = 200, 90, 5, torch.bfloat16
    got = []
    for value, way in ((0.5, "chunks"), (bad, "chunks"), (bad, "walk")):
        if which == "mlstm":
            H, dk, dv = 2, 32, 64
            x, gates = rnd(rows, H * (2 * dk + dv), seed=1).bfloat16().cuda(), (-rnd(rows, 2 * H, seed=2).abs()).float().cuda()
            x[at, 2 * H * dk + col] = value
            y, state = torch.empty(rows, H * dv, device="cuda"), torch.zeros((1, 4 * ops.mlstm_state_floats(H, dk, dv)), dtype=torch.uint8, device="cuda")
            ws = torch.empty(ops.mlstm_workspace_floats(rows, 1, rows, H, dk, dv, bf16), device="cuda") if way == "chunks" else None
            ops.mlstm_scan(y, x[:, :H * dk], x[:, H * dk:2 * H * dk], x[:, 2 * H * dk:], gates, state, 0, i32(0, rows), i32(0), rows, 1, H, dk, dv, 1.0,
                           max_q_len=rows, workspace=ws)
        else:
            R, Q, N, P = 2, 1, 16, 68
            x, dt, one = rnd(rows, R * P + 2 * Q * N, seed=1).bfloat16().cuda(), rnd(rows, R, seed=2).bfloat16().cuda(), torch.ones(R, device="cuda")
            x[at, col] = value
            y, state = torch.empty(rows, R * P, device="cuda"), torch.zeros((1, 4 * ops.ssm_state_floats(R, P, N)), dtype=torch.uint8, device="cuda")
            ws = torch.empty(ops.ssm_workspace_floats(rows, 1, rows, R, N, P, bf16), device="cuda") if way == "chunks" else None
            ops.ssm_scan(y, x, dt, one, one, one, state, 0, i32(0, rows), i32(0), rows, 1, R, Q, N, P, max_q_len=rows, workspace=ws)
        got.append(y)
    good, chunks, walk = got
    # (the column's chunk goes through another loop: the same products, summed one after the other)
    assert rel(chunks[:at], good[:at].double()) < 2e-6
    assert torch.equal(chunks.isfinite(), walk.isfinite()) and not chunks[at:, col].isfinite().any()
    others = torch.arange(y.shape[1], device="cuda") != col
    assert rel(chunks[:, others], good[:, others].double()) < 2e-6


def test_state_space_that_forgets_at_once(ops):
    """A decay of exp(-exp(a_log) dt) with exp(a_log) beyond the floats: every row forgets the ones before it."""
    R, Q, N, P, rows = 2, 1, 16, 8, 130
    xbc, dt = rnd(rows, R * P + 2 * Q * N, seed=3).bfloat16().cuda(), rnd(rows, R, seed=4).bfloat16().cuda()
    one = torch.ones(R, device="cuda")
    got = []
    for ws in (None, torch.full((ops.ssm_workspace_floats(rows, 1, rows, R, N, P, torch.bfloat16),), float("nan"), device="cuda")):
        y = torch.empty(rows, R * P, device="cuda")
        state = torch.zeros((1, 4 * ops.ssm_state_floats(R, P, N)), dtype=torch.uint8, device="cuda")
        ops.ssm_scan(y, xbc, dt, one, 100 * one, one, state, 0, i32(0, rows), i32(0), rows, 1, R, Q, N, P, max_q_len=rows, workspace=ws)
        got.append(y.cpu().double())
    assert bool(torch.isfinite(got[0]).all()) and rel(got[1], got[0]) < 2e-6


def ssm_plain(C, B, x, f, dt, S):
    y = []
    for t in range(len(x)):
        S = torch.exp(f[t]) * S + dt[t] * torch.outer(B[t], x[t])
        y.append(S.t() @ C[t])
    return torch.stack(y), S


@pytest.mark.parametrize("R,Q,N,P", [(8, 2, 128, 64), (3, 1, 20, 36), (2, 2, 4, 8), (4, 2, 260, 132)])
@pytest.mark.parametrize("decay", [-3.0, 1.0, 5.0])
def test_state_space_by_chunks(ops, R, Q, N, P, decay):
    slots, room, C = i32(2, 0, 4, 1, 3), 5, R * P + 2 * Q * N
    state = {way: torch.zeros((room, 64 + 4 * ops.ssm_state_floats(R, P, N)), dtype=torch.uint8, device="cuda") for way in ("chunks", "walk")}
    a_log, bias, skip = (rnd(R, seed=i).float() for i in (1, 2, 3))
    a_log += decay
    plain = [[torch.zeros(N, P, dtype=F64) for _ in range(R)] for _ in range(5)]
    for s, lengths in enumerate(STEPS):
        rows = sum(lengths)
        xbc, dt_in = rnd(rows, C, seed=30 + s).bfloat16(), rnd(rows, R + 3, seed=40 + s).bfloat16()
        xd, dd, cu = xbc.cuda(), dt_in.cuda(), cu_of(lengths)
        floats = ops.ssm_workspace_floats(rows, 5, max(lengths), R, N, P, torch.bfloat16)
        assert floats > 0
        got = {}
        for way in state:
            got[way] = torch.full((rows, R * P), float("nan"), device="cuda")
            ws = torch.full((floats,), float("nan"), device="cuda") if way == "chunks" else None
            ops.ssm_scan(got[way], xd, dd[:, 2:2 + R], bias.cuda(), a_log.cuda(), skip.cuda(), state[way], 64, cu, slots, rows, 5, R, Q, N, P,
                         max_q_len=max(lengths), workspace=ws)
        dt = torch.nn.functional.softplus(dt_in[:, 2:2 + R].double() + bias.double())
        f = -torch.exp(a_log.double()) * dt
        x64, want, r = xbc.double(), torch.empty(rows, R * P, dtype=F64), 0
        for b, n in enumerate(lengths):
            at = slice(r, r + n)
            for h in range(R):
                g = h // (R // Q)
                x = x64[at, h * P:(h + 1) * P]
                y, plain[b][h] = ssm_plain(x64[at, R * P + (Q + g) * N:R * P + (Q + g + 1) * N], x64[at, R * P + g * N:R * P + (g + 1) * N],
                                           x, f[at, h], dt[at, h], plain[b][h])
                want[at, h * P:(h + 1) * P] = y + skip[h].double() * x
            r += n
        e = {way: rel(got[way].cpu(), want) for way in got}
        assert e["chunks"] <= 1.3 * e["walk"] < 1e-5


def chunks_of(lengths):
    return sum(-(-n // 64) for n in lengths)


def mlstm_plain_heads(q, k, v, i, f, state):
    """All heads of a sequence on the device: q, k [T, H, dk], v [T, H, dv], i, f [T, H]; state (S, n, m) is carried on in place."""
    S, n, m = state
    y = torch.empty_like(v)
    for t in range(len(q)):
        new = torch.maximum(f[t] + m, i[t])
        a, b = torch.exp(f[t] + m - new), torch.exp(i[t] - new)
        kt = k[t] * b[:, None]
        S.mul_(a[:, None, None]).baddbmm_(kt[:, :, None], v[t][:, None, :])
        n.mul_(a[:, None]).add_(kt)
        m.copy_(new)
        y[t] = torch.bmm(q[t][:, None, :], S)[:, 0] / (torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6)[:, None]
    return y


@pytest.mark.parametrize("H,dk,dv,lengths", [(64, 512, 256, [130, 500, 900, 70]), (4, 512, 1024, [2100])])
def test_matrix_memory_over_several_windows(ops, H, dk, dv, lengths):
    """More chunks than the workspace holds at once: sequences cut by the edge of a window once, twice and not at all, and a second step
    that goes on from the states. Every row against the recurrence in 64 bits, beside the walk."""
    B, room = len(lengths), 4 * ops.mlstm_state_floats(H, dk, dv)
    slots = i32(*reversed(range(B)))
    state = {way: torch.zeros((B, room), dtype=torch.uint8, device="cuda") for way in ("chunks", "walk")}
    plain = [[torch.zeros(*shape, dtype=F64, device="cuda") for shape in ((H, dk, dv), (H, dk), (H,))] for _ in lengths]
    for s, lens in enumerate((lengths, [70] * B)):
        rows = sum(lens)
        x = rnd(rows, H * (2 * dk + dv), seed=50 + s).bfloat16().cuda()
        gates = torch.cat([rnd(rows, H, seed=60 + s, scale=2.0) - 1.0, -torch.nn.functional.softplus(-(rnd(rows, H, seed=70 + s, scale=2.0) + 3.0))], 1).float().cuda()
        q, k, v = x[:, :H * dk], x[:, H * dk:2 * H * dk], x[:, 2 * H * dk:]
        floats = ops.mlstm_workspace_floats(rows, B, max(lens), H, dk, dv, torch.bfloat16)
        assert s or floats // (H * ((dv + 1) * dk + 6)) < chunks_of(lens)
        got = {}
        for way in state:
            got[way] = torch.full((rows, H * dv), float("nan"), device="cuda")
            ws = torch.full((floats,), float("nan"), device="cuda") if way == "chunks" else None
            ops.mlstm_scan(got[way], q, k, v, gates, state[way], 0, cu_of(lens), slots, rows, B, H, dk, dv, dk ** -0.5, max_q_len=max(lens), workspace=ws)
        x64, g64, r = x.double(), gates.double(), 0
        for b, n in enumerate(lens):
            at = slice(r, r + n)
            want = mlstm_plain_heads(x64[at, :H * dk].reshape(n, H, dk) * dk ** -0.5, x64[at, H * dk:2 * H * dk].reshape(n, H, dk),
                                     x64[at, 2 * H * dk:].reshape(n, H, dv), g64[at, :H], g64[at, H:], plain[b]).reshape(n, H * dv)
            e = {way: rel(got[way][at], want) for way in got}
            # 32-bit sums and exponentials: a few 2^-24
            assert e["chunks"] <= max(2e-6, 1.5 * e["walk"]), (s, b)
            r += n


@pytest.mark.parametrize("R,Q,N,P,lengths", [(64, 8, 256, 256, [130, 1100, 2300, 70])])
def test_state_space_over_several_windows(ops, R, Q, N, P, lengths):
    """The same for the state space, whose chunks hand on S alone."""
    B, C = len(lengths), R * P + 2 * Q * N
    slots, room = i32(*reversed(range(B))), 4 * ops.ssm_state_floats(R, P, N)
    state = {way: torch.zeros((B, room), dtype=torch.uint8, device="cuda") for way in ("chunks", "walk")}
    a_log, bias, skip = (rnd(R, seed=i).float().cuda() for i in (1, 2, 3))
    plain = [torch.zeros(R, N, P, dtype=F64, device="cuda") for _ in lengths]
    for s, lens in enumerate((lengths, [70] * B)):
        rows = sum(lens)
        xbc, dt_in = rnd(rows, C, seed=80 + s).bfloat16().cuda(), rnd(rows, R, seed=90 + s).bfloat16().cuda()
        floats = ops.ssm_workspace_floats(rows, B, max(lens), R, N, P, torch.bfloat16)
        assert s or floats // (R * (P * N + 6)) < chunks_of(lens)
        got = {}
        for way in state:
            got[way] = torch.full((rows, R * P), float("nan"), device="cuda")
            ws = torch.full((floats,), float("nan"), device="cuda") if way == "chunks" else None
            ops.ssm_scan(got[way], xbc, dt_in, bias, a_log, skip, state[way], 0, cu_of(lens), slots, rows, B, R, Q, N, P, max_q_len=max(lens), workspace=ws)
        dt = torch.nn.functional.softplus(dt_in.double() + bias.double())
        keep, x64, r = torch.exp(-torch.exp(a_log.double()) * dt), xbc.double(), 0
        for b, n in enumerate(lens):
            at = slice(r, r + n)
            x = x64[at, :R * P].reshape(n, R, P)
            Bs, Cs = (x64[at, R * P + i * Q * N:R * P + (i + 1) * Q * N].reshape(n, Q, N).repeat_interleave(R // Q, 1) for i in (0, 1))
            S, want = plain[b], torch.empty_like(x)
            for t in range(n):
                S.mul_(keep[r + t][:, None, None]).baddbmm_((Bs[t] * dt[r + t][:, None])[:, :, None], x[t][:, None, :])
                want[t] = torch.bmm(Cs[t][:, None, :], S)[:, 0]
            want += skip.double()[:, None] * x
            e = {way: rel(got[way][at], want.reshape(n, R * P)) for way in got}
            assert e["chunks"] <= max(2e-6, 1.5 * e["walk"]), (s, b)
            r += n


@pytest.mark.parametrize("which", ["mlstm", "ssm"])
def test_short_sequences_of_a_long_step_are_walked(ops, which):
    """Sequences of up to 16 rows beside longer ones have the bits they have alone, rows and states, and no chunk of the workspace; the longer
    ones are the chunks', whatever walks beside them. 70 sequences: the search for a chunk's sequence goes through two turns of 64."""
    bf16, lengths = torch.bfloat16, ([1, 4, 5, 16, 17, 200, 2, 64, 65, 3] * 7)
    B, rows = len(lengths), sum(lengths)
    cu = [0] + torch.tensor(lengths).cumsum(0).tolist()
    if which == "mlstm":
        H, dk, dv = 2, 24, 36
        x, gates = rnd(rows, H * (2 * dk + dv), seed=1).bfloat16().cuda(), (-rnd(rows, 2 * H, seed=2).abs()).float().cuda()
        start = torch.rand((B, ops.mlstm_state_floats(H, dk, dv)), generator=torch.Generator().manual_seed(3)).cuda()
        width, floats = H * dv, lambda *a: ops.mlstm_workspace_floats(*a, H, dk, dv, bf16)

        def scan(at, lens, state, ws):
            y, v = torch.full((sum(lens), width), float("nan"), device="cuda"), x[at]
            ops.mlstm_scan(y, v[:, :H * dk], v[:, H * dk:2 * H * dk], v[:, 2 * H * dk:], gates[at], state, 0, cu_of(lens), i32(*range(len(lens))), sum(lens),
                           len(lens), H, dk, dv, 0.2, max_q_len=max(lens), workspace=ws)
            return y
    else:
        R, Q, N, P = 4, 2, 20, 36
        x, dt = rnd(rows, R * P + 2 * Q * N, seed=1).bfloat16().cuda(), rnd(rows, R, seed=2).bfloat16().cuda()
        one = torch.ones(R, device="cuda")
        start = torch.rand((B, ops.ssm_state_floats(R, P, N)), generator=torch.Generator().manual_seed(3)).cuda()
        width, floats = R * P, lambda *a: ops.ssm_workspace_floats(*a, R, N, P, bf16)

        def scan(at, lens, state, ws):
            y = torch.full((sum(lens), width), float("nan"), device="cuda")
            ops.ssm_scan(y, x[at], dt[at], one, -one, one, state, 0, cu_of(lens), i32(*range(len(lens))), sum(lens), len(lens), R, Q, N, P,
                         max_q_len=max(lens), workspace=ws)
            return y
    bytes_of = lambda t: t.clone().view(torch.uint8)
    state = bytes_of(start)
    room = floats(rows, B, max(lengths))
    assert room > 0
    got = scan(slice(0, rows), lengths, state, torch.full((room,), float("nan"), device="cuda"))
    for b, n in enumerate(lengths[:20]):
        at, alone = slice(cu[b], cu[b + 1]), bytes_of(start[b:b + 1])
        ws = torch.full((floats(n, 1, n),), float("nan"), device="cuda") if n > 96 else None
        y = scan(at, [n], alone, ws)
        if n <= 16 or n > 96:
            assert torch.equal(got[at], y) and torch.equal(state[b], alone[0]), n
        else:
            assert rel(got[at], y.double()) < 2e-6 and rel(state[b].view(torch.float32), alone[0].view(torch.float32).double()) < 2e-6, n
    assert bool(torch.isfinite(got).all())
    # one sequence of 200 rows among 63 of one row: room for its chunks and for those 63 rows could have, not for 63 memories more
    assert 0 < floats(263, 64, 200) <= 5 * floats(200, 1, 200)


def test_what_goes_by_chunks(ops):
    """Short or unknown lengths and 32-bit activations are walked, and so are heads that are no whole fours, whatever workspace is given."""
    bf16 = torch.bfloat16
    assert ops.mlstm_workspace_floats(1000, 2, 64, 4, 64, 64, bf16) == ops.ssm_workspace_floats(1000, 2, 0, 4, 64, 64, bf16) == 0
    assert ops.mlstm_workspace_floats(1000, 2, 65, 4, 64, 64, torch.float32) == ops.ssm_workspace_floats(1000, 2, 65, 4, 64, 64, torch.float32) == 0
    assert ops.mlstm_workspace_floats(1000, 2, 65, 4, 64, 64, bf16) > 0 and ops.ssm_workspace_floats(1000, 2, 65, 4, 64, 64, bf16) > 0
    H, dk, dv, rows = 2, 6, 10, 150
    x, gates = rnd(rows, H * (2 * dk + dv), seed=5).bfloat16().cuda(), (-rnd(rows, 2 * H, seed=6).abs()).float().cuda()
    got = []
    for ws in (None, torch.empty(ops.mlstm_workspace_floats(rows, 1, rows, H, dk, dv, bf16), device="cuda")):
        y = torch.empty(rows, H * dv, device="cuda")
        state = torch.zeros((1, 4 * ops.mlstm_state_floats(H, dk, dv)), dtype=torch.uint8, device="cuda")
        ops.mlstm_scan(y, x[:, :H * dk], x[:, H * dk:2 * H * dk], x[:, 2 * H * dk:], gates, state, 0, i32(0, rows), i32(0), rows, 1, H, dk, dv, 1.0,
                       max_q_len=rows, workspace=ws)
        got.append(y)
    assert torch.equal(*got)


def test_captured_steps_share_the_workspace():
    """Steps of several sizes as graphs, whose chunks lie in one buffer of the engine: it grows between a graph's capture and its replays,
    and every replay gives the logits the step's first, eager run gave."""
    import hector_engine_amd as he
    from hector_engine_amd.registry import config_from_dict
    from tests.test_butolorn_cpu import attn, layer, memory, model, pair
    H, dk, dv = 4, 64, 96
    layers = [layer("parallel", pair(attn(2, 1, 16, 16, 0.25, 8), memory(H, dk, dv, 15.0)), 64)] * 2
    engine = he.Engine(config=config_from_dict(model(layers, 50, 32, 8)), seed=3, dtype="bfloat16", max_tokens=4096, max_slots=2, max_seq_len=1024)
    first, sizes = {}, []
    for n in (100, 100, 300, 100, 500, 300, 200, 100, 500, 300, 200, 100, 500, 200):
        slot = engine.acquire()
        logits = engine.step([he.StepEntry(slot, [(7 * i + n) % 50 for i in range(n)], [0, n // 2, n - 1])]).clone()
        engine.release(slot)
        assert torch.equal(logits, first.setdefault(n, logits)) and bool(torch.isfinite(logits).all())
        sizes.append(engine.shared.buffer.numel())
        engine.scratch.transient((sizes[-1] // 4,), torch.float32).fill_(float("nan"))       # what a graph finds there is not its own
    # 300 and 500 rows run as 512 rows, 200 as 256
    assert engine.stats["step_graph_captures"] == 3 and engine.stats["step_graph_replays"] == 11 and not engine.capture_failures
    assert sizes[1] < sizes[2] == sizes[-1] >= 4 * (512 // 64 + 1) * H * dk * (dv + 1)
