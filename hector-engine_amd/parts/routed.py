"""A routed feed-forward (mixture of experts): each token uses `top` of its experts.

    z = W_router n (+ bias)           fp32, E + I outputs: E experts with weights, then I without
    s = softmax(z)                    over all outputs
    c = s + correction                the choice is made on c, the weights on s
    the outputs are cut into `groups` equal runs of neighbours, each run ranked by the largest c it
    holds; outside the `keep` best runs every c is replaced by -inf; the `top` largest c that are left
    are chosen, and a chosen output weighs s * scale (the weights are not made to sum to one)
    expert e: g = min(W_gate n, limit), u = clamp(W_up n, -limit, limit),
              y = g * sigmoid(alpha g) * (u + 1), result W_down y          (no biases)
    the I outputs without weights are identity experts: their result is n itself
    out = sum over the chosen outputs of weight * result

How it runs: one kernel for the router's product in fp32 (its matrix is kept in 32-bit) and the
choice, and then the experts as one feed-forward: all gate and up rows side by side
in one product, the activation kernel multiplies each expert's stretch by the token's weight for
it (an exact 0 where it was not chosen) and appends weight * n for the identity experts, and one
product with the down matrices side by side (and an identity block) adds everything up. Every step
has the same launches whatever the tokens choose, so it replays as a graph, and a token's sums do
not depend on the rest of the batch. A bfloat16 step of so few rows that they cannot choose more than
half of the experts reads only the chosen experts' rows of the same matrices (ops.chosen_experts). A bfloat16 step of
more than 64 rows sorts its rows by expert and multiplies each expert's matrices with the rows that chose it
(ops.routed_groups) where that is the faster form (_by_expert_times).
Options: `normalize` divides the chosen outputs' weights by their sum (the softmax over the chosen logits
alone; the choice itself is the same, the softmax being monotone); `shared` = {"feed_forward": PartSpec, "name":
suffix of its prefix, "gate": suffix of a stored vector of hidden_size or None} adds an expert that every token
uses, out += sigmoid(gate . n) * shared(n) (gate None: out += shared(n)), the dot product in fp32; `router_bias` adds a
stored number an output to the logits. A shared expert without a gate whose activation is the experts' own joins their
fused matrices as columns of weight 1: it costs no launch of its own.
names: the suffixes of its tensors (router, router_bias, correction; expert e's are 'e<e>.' + gate / up / down).
"""
from __future__ import annotations

import torch

from ..kernels import ops
from .base import BuildEnv, FeedForward, NormedRows, PartSpec, StepContext, TensorSpec, build_part, param, register_part, tensor_name
from .linear import Linear
from .mlp import GatedMLP

# rows whose gate and up columns are held at once in a long prompt step
_ROW_CHUNK = 4096


def _linears(part) -> list[Linear]:
    """The linear layers of a bound part and of the parts it is made of."""
    own = [v for v in vars(part).values() if isinstance(v, Linear)]
    return own + [lin for child in part.children() for lin in _linears(child)]


@register_part("feed_forward", "routed_experts")
class RoutedExperts(FeedForward):
    routes = True

    def __init__(self, params: dict, prefix: str, env: BuildEnv):
        super().__init__(prefix, env)
        self.hidden = param(params, "hidden_size", int)
        self.inter = param(params, "intermediate_size", int)
        self.real = param(params, "experts", int)
        self.identity = param(params, "identity_experts", int, 0)
        self.top = param(params, "top", int)
        self.scale = param(params, "scale", float, 1.0)
        self.groups = param(params, "groups", int, 1)
        self.keep = param(params, "keep_groups", int, self.groups)
        self.has_correction = param(params, "correction", bool, True)
        self.normalize = param(params, "normalize", bool, False)
        self.has_bias = param(params, "router_bias", bool, False)
        self.bias = None
        shared = param(params, "shared", dict, None)
        self.shared = self.shared_gate = self._shared_gate = None
        if shared:
            self.shared = build_part("feed_forward", shared["feed_forward"], prefix + shared.get("name", "shared") + ".", env)
            if shared.get("gate"):
                self._shared_gate = prefix + shared.get("name", "shared") + "." + shared["gate"]
        self.limit = param(params, "limit", float, 0.0)
        self.alpha = param(params, "alpha", float, 1.702 if self.limit > 0 else 1.0)
        self.up_shift = param(params, "up_shift", float, 1.0 if self.limit > 0 else 0.0)
        # columns of a shared expert that run as part of the experts' own products
        act = {"alpha": self.alpha, "limit": self.limit, "up_shift": self.up_shift, "cubic": 0.0}
        self.shared_cols = 0
        if isinstance(self.shared, GatedMLP) and not self._shared_gate \
                and {**{"alpha": 1.0, "limit": 0.0, "up_shift": 0.0, "cubic": 0.0}, **self.shared.act} == act:
            self.shared_cols = self.shared.inter
        # rows prepared for a norm may come as they are, where they owe nothing
        self.accepts_normed_rows = self.shared is None or self.shared_cols > 0
        E = self.real + self.identity
        if self.real <= 0 or self.identity < 0 or self.inter <= 0:
            raise ValueError("routed_experts: experts and intermediate_size must be positive, identity_experts not negative")
        if self.groups <= 0 or E % self.groups or not 0 < self.keep <= self.groups:
            raise ValueError(f"routed_experts: {E} router outputs do not form {self.groups} equal groups "
                             f"of which {self.keep} are kept")
        if not 0 < self.top <= self.keep * (E // self.groups):
            raise ValueError(f"routed_experts: top {self.top} exceeds the {self.keep * (E // self.groups)} outputs "
                             "of the kept groups")
        names = param(params, "names", dict, {})
        self._router = tensor_name(prefix, names, "router", "router.weight")
        self._correction = tensor_name(prefix, names, "correction", "router.correction")
        self._bias = tensor_name(prefix, names, "router_bias", "router.bias")
        self._expert = names.get("expert", "experts.{e}.")
        self._sub = {k: names.get(k, d) for k, d in (("gate", "gate_proj.weight"), ("up", "up_proj.weight"),
                                                     ("down", "down_proj.weight"))}
        self.router: torch.Tensor | None = None
        self.correction = None
        self.gate_up: Linear | None = None
        self.down: Linear | None = None

    def _name(self, e: int, which: str) -> str:
        return self.prefix + self._expert.format(e=e) + self._sub[which]

    def tensor_specs(self):
        specs = {self._router: TensorSpec((self.real + self.identity, self.hidden))}
        if self.has_correction:
            specs[self._correction] = TensorSpec((self.real + self.identity,))
        if self.has_bias:
            specs[self._bias] = TensorSpec((self.real + self.identity,), ("normal", 0.1))
        for e in range(self.real):
            specs[self._name(e, "gate")] = TensorSpec((self.inter, self.hidden))
            specs[self._name(e, "up")] = TensorSpec((self.inter, self.hidden))
            specs[self._name(e, "down")] = TensorSpec((self.hidden, self.inter))
        if self.shared is not None:
            specs.update(self.shared.tensor_specs())
        if self._shared_gate:
            specs[self._shared_gate] = TensorSpec((1, self.hidden))
        return specs

    def children(self):
        return [self.shared] if self.shared is not None else []

    def bind(self, tensors):
        # the router's sums are 32-bit whatever the run's precision: its matrix is kept in float32
        self.router = tensors[self._router].to(torch.float32).contiguous()
        self.correction = tensors[self._correction] if self.has_correction else None
        self.bias = tensors[self._bias] if self.has_bias else None
        gu, downs = [], []
        for e in range(self.real):
            g, u = tensors.pop(self._name(e, "gate")), tensors.pop(self._name(e, "up"))
            # gate i of an expert at row 2i of its stretch, its up at 2i + 1
            gu.append(torch.stack([g, u], 1).reshape(2 * self.inter, self.hidden))
            downs.append(tensors.pop(self._name(e, "down")))
        if self.shared_cols:
            g, u, dn = (tensors.pop(self.shared._names[k]) for k in ("gate", "up", "down"))
            gu.append(torch.stack([g, u], 1).reshape(2 * self.shared_cols, self.hidden))
            downs.append(dn)
        if self.identity:
            # the identity experts' share rides through the down product on an identity block
            downs.append(torch.eye(self.hidden, dtype=downs[0].dtype, device=downs[0].device))
        self.gate_up = Linear(torch.cat(gu, 0).contiguous())
        self.down = Linear(torch.cat(downs, 1).contiguous())
        if self.shared is not None and not self.shared_cols:
            self.shared.bind(tensors)
            for lin in _linears(self.shared):
                lin.one_round_tiles = False                # (the router may read rows no norm has evened out)
        if self._shared_gate:
            self.shared_gate = tensors[self._shared_gate].reshape(-1).contiguous()

    def _few_rows(self, rows: int, x, ctx: StepContext) -> bool:
        """Whether the step runs through the chosen experts alone (kernels.ops.chosen_experts): bfloat16 with the
        fast kernels, sizes in multiples of 8, and so few rows that they cannot choose more than half of the
        experts. (The 32-bit path keeps the products over all experts, whose sums do not depend on the batch.)"""
        return (ctx.env.fast_kernels and ctx.env.dtype == torch.bfloat16 and self.gate_up.weight.dtype == torch.bfloat16
                and self.inter % 8 == 0 and self.shared_cols % 8 == 0 and self.hidden % 8 == 0 and 2 * rows * self.top <= self.real)

    def _leaves_out(self, rows: int) -> tuple[bool, bool]:
        """Whether the products over all experts of a step of up to 16 bfloat16 rows, the first and the second, leave out the experts that
        nobody chose (routed_act gives exact zeros for those). Every workgroup asks for the choice before its weights, 2 us and more a
        product: 1.04 to 1.3 of its time where every expert is chosen. So only where the experts expected without a row (`top` even among the
        outputs) are a quarter and 80 MB of the first product's weights, in rows of 1024 and more, and a fifth of 50 MB and more of the
        second's (whose groups of k are no shorter than 512, a turn of the kernel's walk). Over 13,700 random sizes with weights from
        memory (4 to 64 experts of 256 to 4096, 2 to 16 rows of 512 to 4096) the 1731 first products that this takes need 0.78 of the time of
        the whole ones in the geometric mean, 5 of them 1.03 to 1.07, the 3236 second ones 0.85, none above 1.03; all others 1.12 and 1.04 of it. 4 rows
        of 2048, 4 chosen of 16 experts of 2048: 49.3 us and 41.5, 33.5 and 29.9."""
        unused = (1 - self.top / (self.real + self.identity)) ** rows
        mb = 2e-6 * self.real * self.inter * self.hidden
        return (self.hidden >= 1024 and unused >= 0.25 and unused * 2 * mb >= 80, self.inter >= 512 and unused >= 0.2 and mb >= 50)

    def _many_rows(self, rows: int, x, ctx: StepContext) -> int:
        """The rows a tile has where the step runs expert by expert over the rows that chose it (kernels.ops.routed_groups),
        0 where it runs through the products over all experts. For bfloat16 with the fast kernels, sizes in multiples
        of 64, no shared columns, and a choice of half of the experts at most, from 65 rows on (fewer go through the kernels
        that carry norms), where _by_expert_times expects the faster of the two tile heights in 0.8 of the other form's time."""
        turn = min(rows, _ROW_CHUNK)
        if not (ctx.env.dtype == torch.bfloat16 and isinstance(x, torch.Tensor) and not self.shared_cols
                and 2 * self.top <= self.real <= 1024 and self.inter % 64 == 0 and self.hidden % 64 == 0
                and not (self.shared is not None and self.identity) and ops.tiles_read(x)
                # (a lane's offsets into the rows and into 256 rows of a weight are 32-bit)
                and 2 * max(turn * self.hidden, 256 * (self.real * self.inter + self.hidden)) < 1 << 32
                and self.gate_up.own_tiles(turn, ctx) and (self.shared is not None or self.down.own_tiles(turn, ctx))):
            return 0
        low, high, over_all = self._by_expert_times(turn)
        return 0 if min(low, high) > 0.8 * over_all else 128 if low <= high else 256

    def _by_expert_times(self, rows: int) -> tuple[float, float, float]:
        """Microseconds the experts of so many rows are expected to take: by expert in tiles of 128 and of 256 rows, and as products over
        all experts. A round of tiles on the chip costs a start and its stages of 64 k, an expert has whole tiles however few rows
        chose it, every choice's part of the sum is written and read in 32 bits, and sorting takes a nanosecond a choice; the
        library's products cost their operations or their weights' bytes. The numbers were fitted with the tile kernel that had eight
        wavefronts; with the one there is they are 1.03 and 1.04 of what by-expert steps take (0.9 beside a shared expert) and 0.92 of the products
        over all, each off by a fifth (standard deviation over 2709 random sizes, 2 to 256 experts of 64 to 4096, 65 to 4096 rows of 256
        to 7168). With the factor 0.8 the 1403 of these that go by expert take 0.43 of the other form's time in the geometric mean, 5 of
        them 1.03 to 1.05 (beside a shared expert 1323, 0.72, 4 of them 1.03 to 1.11), in tiles that are 1.006 of the better of the
        two heights: 16 experts of 2048 over rows of 2048, 4 chosen, 65 rows 118 us beside 115, 512 150 beside 220, 2048 318 beside 874.
        Few or small experts are left to the other form: 2 of 64 over 224 rows of 1728, 1 chosen, 13 us beside 44; 201 of the 1306 left would
        be below 0.8 by expert."""
        D, I, real = self.hidden, self.inter, self.real
        choices, cus = rows * self.top, ops.compute_units()

        def library(cols: int, k: int) -> float:
            return max(2 * rows * cols * k / 1300e6, 2 * cols * k / 4e6)

        def by_expert(bm: int, start: float, begin: float, stage: float) -> float:
            tiles = min(min(real, choices) * -(-choices // (real * bm)), choices // bm + min(choices, real))

            def rounds(cols: int, k: int) -> float:
                return -(-tiles * -(-cols // 256) // cus) * (begin + k // 64 * stage)
            first = start + choices / 1000 + rounds(2 * I, D)
            if self.shared is not None:      # (the second product stays one over all experts, over rows cleared first)
                return first + 2 * rows * real * I / 0.8e6 + library(D, real * I)
            return first + rounds(D, I) + 4 * choices * D / 2e6
        over_all = 14 + library(2 * real * I, D) + library(D, real * I) + 6 * rows * real * I / 1.5e6
        return by_expert(128, 9, 7.5, 0.9), by_expert(256, 11, 10.5, 1.33), over_all

    def _by_expert(self, x, dense, ids, weights, rows: int, bm: int, act: dict, ctx: StepContext):
        out = ctx.alloc((rows, self.hidden))
        for r0 in range(0, rows, _ROW_CHUNK):
            n = min(_ROW_CHUNK, rows - r0)
            turn = ctx.scratch.mark()
            ints, slots = ops.routed_groups_sizes(n, self.top, self.real, bm)
            lists = ctx.alloc((ints,), torch.int32)
            if self.shared is not None:
                # Beside a shared expert the sum over the experts stays one product over all of them, with its order of
                # sums: a design that routes rows as they are, without a norm, turns near ties over at any change of it
                # (Domorax: 3 to 6 % of the logits; with the first product alone by expert they stay bit for bit what they were).
                h = ctx.alloc((n, self.real * self.inter)).zero_()
                ops.routed_groups_act(h, lists, x[r0:r0 + n], self.gate_up.weight, ids[r0:r0 + n], weights[r0:r0 + n], n,
                                      self.real, self.inter, bm=bm, **act)
                self.down(h, n, ctx, out=out[r0:r0 + n])
                ctx.scratch.release(turn)
                continue
            h = ctx.alloc((slots, self.inter))
            partial = ctx.alloc((n * self.top, self.hidden), torch.float32)
            ops.routed_groups(out[r0:r0 + n], lists, h, partial, x[r0:r0 + n], self.gate_up.weight, self.down.weight,
                              ids[r0:r0 + n], weights[r0:r0 + n], dense[r0:r0 + n], n, self.real, self.inter, bm=bm, **act)
            ctx.scratch.release(turn)
        return out

    def forward(self, x, ctx: StepContext):
        if self.shared is None or self.shared_cols:
            return self._routed(x, ctx, True)
        rows = ctx.rows
        routed = self._routed(x, ctx, False)
        common = self.shared.forward(x, ctx)
        out = ctx.alloc((rows, self.hidden))
        if self.shared_gate is not None:
            ops.gated_add(out, routed, common, x, self.shared_gate, rows)
        else:
            ops.scaled_sum(out, routed, common, rows, 1.0, 1.0)
        return out

    def _routed(self, x, ctx: StepContext, may_sink: bool):
        rows, real, I, S = ctx.rows, self.real, self.inter, self.shared_cols
        # rows a product has left for this norm: read as they lie where they owe nothing (and no identity expert wants
        # them row by row), else made into a tensor, by the router's launch where that pays and its reads are whole
        pieces = isinstance(x, NormedRows) and x.finished and x.pieces and not self.identity
        owed = None
        given, read, read_pieces = x, x, pieces      # what the experts' first product reads, and the router
        if isinstance(x, NormedRows):
            read, read_pieces = x.scaled, x.pieces
            if pieces:
                x = x.scaled
            elif self.router.shape[0] <= 64 and x.dim % 8 == 0 and read.data_ptr() % 16 == 0 and self.router.data_ptr() % 16 == 0:
                given = ctx.alloc((rows, x.dim), read.dtype)
                owed = (x.partials, x.eps, given)
                x = given
            else:
                given = read = x = x.tensor(ctx)
                read_pieces = False
        dense = ctx.alloc((rows, real + 1), torch.float32)
        ids = ctx.alloc((rows, self.top), torch.int32)
        weights = ctx.alloc((rows, self.top), torch.float32)
        # the router's product (fp32 sums over the rows as they are) and the choice, one launch
        ops.route_tokens(dense, ids, weights, None, self.correction, rows, real, self.groups, self.keep,
                         self.top, self.scale, x=read, router=self.router, normalize=self.normalize, bias=self.bias,
                         x_pieces=read_pieces, owed=owed)
        cols = real * I + S + (self.hidden if self.identity else 0)
        act = {"alpha": self.alpha, "limit": self.limit, "up_shift": self.up_shift}
        if self._few_rows(rows, x, ctx):
            # the rows of the step choose at most half of the experts: only those experts' weights are read
            h = ctx.alloc((rows * (self.top * I + S),))
            out = ctx.alloc((rows, self.hidden))
            ops.chosen_experts(out, h, x, self.gate_up.weight, self.down.weight, ids, weights, dense, rows, real, I,
                               shared=S, x_pieces=pieces, **act)
            return out
        bm = self._many_rows(rows, x, ctx)
        if bm:
            return self._by_expert(x, dense, ids, weights, rows, bm, act, ctx)
        if rows <= _ROW_CHUNK:
            first, second = self._leaves_out(rows)
            gu = self.gate_up(given, rows, ctx, used=(dense, real, 2 * I, False) if first else None)
            h = ctx.alloc((rows, cols))
            ops.routed_act(h, gu, dense, x if self.identity else None, rows, real, I, shared=S, **act)
            return self.down(h, rows, ctx, sink=ctx.take_sink() if may_sink else None,
                             used=(dense, real, I, True) if second else None)
        out = ctx.alloc((rows, self.hidden))
        for r0 in range(0, rows, _ROW_CHUNK):
            n = min(_ROW_CHUNK, rows - r0)
            turn = ctx.scratch.mark()
            gu = self.gate_up(x[r0:r0 + n], n, ctx)
            h = ctx.alloc((n, cols))
            ops.routed_act(h, gu, dense[r0:r0 + n], x[r0:r0 + n] if self.identity else None, n, real, I, shared=S,
                           **act)
            self.down(h, n, ctx, out=out[r0:r0 + n])
            ctx.scratch.release(turn)
        return out
