"""The linear layer all parts share: y[M,N] = x[M,K] . W[N,K]^T (+ bias).

Which kernel runs is looked up in the table of kernel routes (kernels.routes) under
("linear", (weight dtype, activation dtype)) with the step's row count; the routes this file
registers:
  float32 weights          -> the plain FMA kernel (fixed summation order per element);
                              a weight that was stored in 32-bit stays 32-bit and runs
                              through it also under bfloat16 activations
  bfloat16, M <= 16        -> the block-split MFMA kernel: K is cut inside the workgroup,
                              one launch gives the finished result
  bfloat16, 17 <= M <= 64  -> the MFMA kernel that shares the activation rows of a workgroup
                              through LDS (kernels.ops.gemm_rows); products with few weight rows
                              are cut along K across workgroups and leave fp32 slices, which a
                              small kernel adds (into the result, or straight into the residual)
  bfloat16, M > 64         -> the library matrix product (the reference calls its BLAS
                              library for every product: kernels/matmul_cublas.cu:240-277), or
                              the tiles of kernels.ops.gemm_tall or gemm_few_tiles where they are faster
                              (_long, tall_gated, gated_tile, _few_tiles)
  fp32 results (logits)    -> the MFMA kernels up to 64 rows, above that the library,
                              which writes fp32 from bf16 operands

Both MFMA kernels carry an RMS norm across a pair of products, so that a step of up to 64
rows has no norm kernels: given a :class:`ResidualSink` the product adds its result
to the residual rows itself and leaves r * gain and the sums of r^2 for the norm that
follows (:class:`NormedRows`); given NormedRows as input it applies the owed row scale
to its sums. Any other path turns NormedRows into a tensor first and ignores the sink.

Between such products the bf16 rows travel piece-major (kernels.ops.pieces_shape): an
operand load then touches two cache lines instead of sixteen (at the Qwen2.5-7B shapes 2 us a
layer at 8 rows, 10 us at 16; at 64 rows the gated product takes 61 us against 97 us). The
rows a product leaves for the next norm are written so; a producer of its input (attention,
the gated product) writes so after asking reads_pieces().
"""
from __future__ import annotations

from dataclasses import dataclass

import torch

from ..kernels import library_tuning, ops, profiler, routes
from .base import NormedRows, PieceRows, ResidualSink, StepContext

BF16, F32 = torch.bfloat16, torch.float32


@dataclass(frozen=True)
class ProductCase:
    """What a route of "linear" decides by."""
    rows: int
    N: int
    K: int
    fast: bool          # the environment allows the MFMA kernels and the library


def _operand(x):
    """(activation dtype, the tensor a kernel reads, the owed row scale or None, whether
    that tensor lies piece-major) of a tensor, NormedRows or PieceRows."""
    if isinstance(x, NormedRows):
        return x.scaled.dtype, x.scaled, (x.partials, x.eps), x.pieces
    if isinstance(x, PieceRows):
        return x.pieces.dtype, x.pieces, None, True
    return x.dtype, x, None, False


class Linear:
    def __init__(self, weight: torch.Tensor, bias: torch.Tensor | None = None):
        if weight.dim() != 2:
            raise ValueError("Linear weight must be [out, in]")
        self.weight = weight
        self.bias = bias
        self.out_features, self.in_features = weight.shape
        self.one_round_tiles = False        # set by a part: _long's, gated_tile's and K slices' products may run in tiles of this library's own
        self.ordered = False                # set by the model: the few-rows product keeps an older order of sums (ops.gemm_blocksplit)
        self._plans: dict[bool, tuple[int, int]] = {}
        self._chosen: dict[tuple, routes.Route] = {}     # (rows, activations, fast) -> route, for one version of the table
        self._chosen_version = -1

    def route(self, rows: int, ctx: StepContext, act: torch.dtype) -> routes.Route:
        """The kernel route of this product at this many rows of this activation dtype (remembered
        per row count while the table of routes does not change: a step asks a hundred times)."""
        if self._chosen_version != routes.version() or len(self._chosen) > 256:
            self._chosen.clear()
            self._chosen_version = routes.version()
        key = (rows, act, ctx.env.fast_kernels)
        route = self._chosen.get(key)
        if route is None:
            N, K = self.weight.shape
            route = routes.choose("linear", (self.weight.dtype, act), ProductCase(rows, N, K, ctx.env.fast_kernels))
            self._chosen[key] = route
        return route

    def own_tiles(self, rows: int, ctx: StepContext, act: torch.dtype = BF16) -> bool:
        """Whether a part may run this many rows through the tile kernels itself (kernels.ops.gemm_tall, routed_groups): where
        the library's route would, so that a route registered in front of it still gets its products."""
        return bool(routes.routes_of("linear", (self.weight.dtype, act))) and self.route(rows, ctx, act).run is Linear._run_library

    def _has(self, trait: str, rows: int, ctx: StepContext, act: torch.dtype) -> bool:
        if not routes.routes_of("linear", (self.weight.dtype, act)):
            return False
        return trait in self.route(rows, ctx, act).traits

    def reads_pieces(self, rows: int, ctx: StepContext) -> bool:
        """Whether bf16 input rows may come piece-major (PieceRows)."""
        return self._has("pieces", rows, ctx, BF16)

    def k_slices(self, x, rows: int, ctx: StepContext):
        """The product without bias as the fp32 sums of its K slices, [slices, rows, N], where the
        kernel of this step cuts it along K across workgroups (17 to 64 rows of a weight with few
        rows); None where it does not, and the caller calls the layer as usual. A reader that adds
        the slices itself, in their order, and rounds to the activation dtype has the bits the
        layer's own sum would have written, and saves that launch."""
        act, a, scale, pieces = _operand(x)
        if rows <= ops.BLOCKSPLIT_PIECES_MAX_M or not self._has("k_slices", rows, ctx, act):
            return None
        splits = self._plan(rows)[1]
        if splits == 1:
            return None
        partial = ctx.alloc((splits, rows, self.weight.shape[0]), torch.float32)
        ops.gemm_rows(None, partial, a, self.weight, None, rows, row_scale=scale, x_pieces=pieces)
        return partial

    def _plan(self, rows: int) -> tuple[int, int]:
        """(workgroups along N, K slices) of the 17-to-64-row kernel for this weight."""
        key = rows <= 32
        if key not in self._plans:
            self._plans[key] = ops.gemm_rows_plan(rows, *self.weight.shape)
        return self._plans[key]

    def __call__(self, x, rows: int, ctx: StepContext, *, use_bias: bool = True,
                 out_dtype: torch.dtype | None = None, out: torch.Tensor | None = None,
                 sink: ResidualSink | None = None, used=None):
        """x: a tensor, NormedRows or PieceRows. With a sink the result may go into the
        residual stream directly; the call then returns None. used: groups of the weight that may be left out
        (ops.gemm_blocksplit), where the kernel can."""
        bias = self.bias if use_bias else None
        act = _operand(x)[0]
        if used is not None and 0 < rows <= ops.BLOCKSPLIT_PIECES_MAX_M and self.route(rows, ctx, act).run is Linear._run_mfma \
                and (out_dtype or act) == BF16:
            return self._run_mfma(x, rows, ctx, bias, BF16, out, sink, used)
        return self.route(rows, ctx, act).run(self, x, rows, ctx, bias, out_dtype or act, out, sink)

    # ---- the routes' bodies ----

    def _run_mfma(self, x, rows, ctx, bias, out_dtype, out, sink, used=None):
        """Up to 64 rows of bf16: the block-split kernel (up to 16 rows) or the rows kernel."""
        w = self.weight
        N = w.shape[0]
        act, a, scale, pieces = _operand(x)
        # (up to 16 rows the residual epilogue has one order of sums, not the kept one)
        if sink is not None and out is None and out_dtype == act and not (self.ordered and rows <= ops.BLOCKSPLIT_PIECES_MAX_M) \
                and sink.stream.rows == rows and sink.stream.resid.shape[-1] == N:
            return self._into_residual(x, bias, rows, ctx, sink, used)
        if out is None:
            out = ctx.alloc((rows, N), out_dtype)
        if rows <= ops.BLOCKSPLIT_PIECES_MAX_M:
            ops.gemm_blocksplit(out, a, w, bias, rows, row_scale=scale, x_pieces=pieces, used=used, ordered=self.ordered)
            return out
        splits = self._plan(rows)[1]
        if splits == 1:
            ops.gemm_rows(out, None, a, w, bias, rows, row_scale=scale, x_pieces=pieces)
            return out
        partial = ctx.alloc((splits, rows, N), torch.float32)
        ops.gemm_rows(None, partial, a, w, None, rows, row_scale=scale, x_pieces=pieces)
        ops.splitk_reduce(out, partial, bias, rows, splits)
        return out

    def _dense(self, x, rows, ctx, out_dtype, out):
        """(x as a plain tensor, the result buffer) for the routes that read row-major rows."""
        if isinstance(x, PieceRows):
            raise TypeError("Linear: piece-major rows for a product that does not read them (ask reads_pieces)")
        if isinstance(x, NormedRows):
            x = x.tensor(ctx)
        if out is None:
            out = ctx.alloc((rows, self.weight.shape[0]), out_dtype)
        return x, out

    def _run_plain(self, x, rows, ctx, bias, out_dtype, out, sink):
        """The plain kernel (fixed summation order) in the precision of its operands."""
        x, out = self._dense(x, rows, ctx, out_dtype, out)
        if rows == 0:
            return out
        if x.dtype == torch.float32 and out_dtype != torch.float32:
            raise TypeError("float32 activations give float32 outputs")
        self._plain(out, x, bias, rows, ctx)
        return out

    def _run_plain_widened(self, x, rows, ctx, bias, out_dtype, out, sink):
        """A weight kept in 32-bit under bfloat16 activations: the rows widened, the plain kernel."""
        x, out = self._dense(x, rows, ctx, out_dtype, out)
        if rows == 0:
            return out
        N, K = self.weight.shape
        x32 = ctx.alloc((rows, K), torch.float32)
        x32.copy_(x[:rows])
        y32 = out if out_dtype == torch.float32 else ctx.alloc((rows, N), torch.float32)
        self._plain(y32, x32, bias, rows, ctx)
        if y32 is not out:
            out[:rows].copy_(y32)
        return out

    def _run_library(self, x, rows, ctx, bias, out_dtype, out, sink):
        x, out = self._dense(x, rows, ctx, out_dtype, out)
        if rows == 0:
            return out
        if library_tuning.enabled() and not library_tuning.worth_tuning(rows):
            with library_tuning.no_new_tuning():
                return self._library(x, bias, rows, out, out_dtype, ctx)
        return self._library(x, bias, rows, out, out_dtype, ctx)

    def _plain(self, out, x, bias, rows: int, ctx: StepContext) -> None:
        """The plain product (fixed summation order); some products of few rows want a workspace for their segment sums."""
        floats = ops.gemm_plain_workspace_floats(rows, *self.weight.shape, a=x, w=self.weight, out=out)
        ws = ctx.alloc((floats,), torch.float32) if floats else None
        ops.gemm_plain(out, x, self.weight, bias, rows, workspace=ws)

    def _library_slices(self, rows: int) -> int:
        """K slices for the library's product of a long-K weight with few output columns at up to
        512 rows (the down projection in a step of a few hundred tokens): the library's tiles of
        256 x 256 outputs would be a dozen or two for a chip of 256 compute units, each walking all
        of K. As a batched product over K slices with fp32 results, which he_splitk_reduce adds
        in slice order, the Qwen2.5-7B down projection takes 58 us instead of 99 at 128 rows, 50
        instead of 122 at 200, 54 instead of 126 at 256, 80 instead of 197 at 512 (four slices); the
        Qwen2.5-32B one 68 instead of 180 at 128 rows, the Qwen2-72B one (four slices) 142 instead of 226. Products with
        K below 8192 gain nothing (q||k||v, o, gate||up: measured)."""
        N, K = self.weight.shape
        if rows > 512 or K < 8192 or K < 3 * N:
            return 1
        tiles = -(-rows // 256) * -(-N // 256)
        slices = 8 if tiles <= 20 else 4 if tiles <= 40 else 2 if tiles <= 64 else 1
        while slices > 1 and K % (8 * slices):
            slices //= 2
        return slices

    def _tile_fill(self, rows: int, slices: int = 1) -> tuple[float, float]:
        """Of the tile gemm_tall_tile chooses (for so many K slices): the share of its rounds of the chip that has tiles, and that has real outputs (none of no rows)."""
        if rows == 0:
            return 0.0, 0.0
        N, K = self.weight.shape
        bm, bn = ops.gemm_tall_tile(rows, N, K, slices)
        tiles, cus = -(-rows // bm) * -(-N // bn) * slices, ops.compute_units()
        places = -(-tiles // cus) * cus
        return tiles / places, rows * N * slices / (places * bm * bn)

    def _long(self, rows: int, x, out, out_dtype) -> bool:
        """Whether a product of long K runs in tiles of this library's own (kernels.ops.gemm_tall): for K from 16448 to 27648, where
        the library's default choice drops to 0.65 to 0.9 PFLOP/s at many sizes (from 1.0 to 1.4 at shorter K), and tiles of gemm_tall_tile's
        choice that leave at most 0.3 of their rounds without real outputs. Over 468 products of 458 to 12032 rows and 480 to 12892
        columns 0.53 to 1.11 of the library's time, 0.76 in the geometric mean, 25 of them above 1.03 (2048 x 3584 x 18944 230 us, the library 358; 12001 rows
        1144, 1528). Not where the library's own tiles of 256 x 256 are one or two rounds all but whole, which it runs at 1.4 to 1.55 PFLOP/s (37 such
        products, 1.07 of its time in the geometric mean: 4608 x 3584 x 18944 450 us, 404), nor several rounds of tiles of 128 x 256, which
        reach 1.1 to 1.2 (17 products, 0.68 to 1.19: 6889 x 3584 x 18944 803 us, 692); with 0.4 to 0.6 of the rounds real up to 1.19, with less up to 3. At K up to 16384 the library's choice is as often
        as not the faster one (0.57 to 1.24 of its time over 300 products of whole rounds, 0.98 in the geometric mean), and beyond K 27648 too
        (8192 x 29568 up to 1.24). Only where a part allows it (one_round_tiles): the library adds some tiles of such a product in
        two halves, so 6 results in 10,000 differ in their last bit, which a router over rows that no norm has evened out turns into
        other choices."""
        N, K = self.weight.shape
        return not library_tuning.enabled() and self.one_round_tiles and out_dtype == BF16 and 16384 < K <= 27648 and K % 64 == 0 \
            and N % 4 == 0 and x.is_contiguous() and out.is_contiguous() and self.weight.is_contiguous() and ops.tiles_read(x, self.weight, out) \
            and self._tile_fill(rows)[1] >= 0.7 and not (0.925 <= self._rounds(rows, 256) <= 1 or 1.93 <= self._rounds(rows, 256) <= 2) \
            and (self._rounds(rows, 128) <= 1 or ops.gemm_tall_tile(rows, N, K) != (128, 256))

    def _slices_in_tiles(self, rows: int, slices: int, x) -> bool:
        """Whether the K slices of a product of up to 512 rows (_library_slices) run in this library's own tiles: more than 2048 columns, and
        tiles for 0.7 of a round of the chip or more. Over 90 products that this takes 0.67 to 1.04 of the batched product's time and its sum,
        0.89 in the geometric mean (203 x 3584 x 18944 45.9 us beside 48.8 without the sum); of 70 others 0.65 to 1.86, 1.06 in the
        mean (128 x 2048 x 27648 49.7 and 38.3, 292 x 2048 x 8192 27.0 and 24.5, 78 x 496 x 27648 38.6 and 20.8). Only where a part allows it
        (see _long): of 310 products of 65 to 512 rows 295 had the library's bits, 15 of some widths (768 x 16384 at 65 rows,
        2192 x 28672 at 128) 3 results in 10,000 that differ in their last bit."""
        N, K = self.weight.shape
        return self.one_round_tiles and not library_tuning.enabled() and N > 2048 and N % 4 == 0 and K % (64 * slices) == 0 \
            and self.weight.is_contiguous() and ops.tiles_read(x, self.weight) and self._tile_fill(rows, slices)[0] >= 0.7

    def _few_tiles(self, rows: int, x, out, out_dtype) -> int:
        """The tile (kernels.ops.few_tiles_tile) of a product whose tiles are one round of the chip, 0 where the library runs it: tiles of
        at most 208 rows and columns together, for half of the chip's units or more, of K up to 5120; of K up to 1024
        whatever their number. 256 rows of 4608 x 3584 take 22 us, the library 36.7; over 262 random products that this takes
        (65 to 1200 rows) 0.70 of the library's time in the geometric mean, one above 1.04 of it (593 rows of 3164 x 4096, 1.10).
        Fewer tiles of a longer K (up to 1.9 of it), K beyond 5120 (up to 1.4) and larger tiles (up to 1.3) stay with the library, which cuts such
        products along K. The sums are the library's where it does not cut: 260 of the 262 gave its bits."""
        N, K = self.weight.shape
        if library_tuning.enabled() or not (out_dtype == BF16 and K <= 5120 and K % 64 == 0 and N % 4 == 0 and x.is_contiguous()
                                            and out.is_contiguous() and self.weight.is_contiguous()
                                            and ops.tiles_read(x, self.weight, out)):
            return 0
        tile = ops.few_tiles_tile(rows, N)
        bm, bn = tile >> 16, tile & 0xffff
        if tile == 0 or bm + bn > 208 or (K > 1024 and 2 * -(-rows // bm) * -(-N // bn) < ops.compute_units()):
            return 0
        return tile

    def _library(self, x, bias, rows, out, out_dtype, ctx):
        """More than 64 rows: the library's product, or tiles of this one's own; it also writes fp32 results (the logits) from
        bf16 operands (the head of the Qwen2.5-7B shape at 64 rows: 217 us)."""
        w = self.weight
        if self._long(rows, x, out, out_dtype):
            bm, bn = ops.gemm_tall_tile(rows, *w.shape)
            ops.gemm_tall(out, x, w, bias, rows, bm=bm, bn=bn)
            return out
        tile = self._few_tiles(rows, x, out, out_dtype)
        if tile:
            ops.gemm_few_tiles(out, x, w, bias, rows, tile)
            return out
        slices = self._library_slices(rows) if out_dtype == torch.bfloat16 and x.is_contiguous() else 1
        if slices > 1:
            N, K = w.shape
            partial = ctx.alloc((slices, rows, N), torch.float32)
            if self._slices_in_tiles(rows, slices, x):
                bm, bn = ops.gemm_tall_tile(rows, N, K, slices)
                ops.gemm_tall(partial, x, w, None, rows, bm=bm, bn=bn, slices=slices)
                ops.splitk_reduce(out, partial, bias, rows, slices)
                return out
            with profiler.span("library_gemm"):
                # views, no copies: slice s of x is [rows, K / slices] at row stride K, of w likewise
                torch.bmm(x[:rows].view(rows, slices, K // slices).transpose(0, 1),
                          w.view(N, slices, K // slices).permute(1, 2, 0),
                          out_dtype=torch.float32, out=partial)
            ops.splitk_reduce(out, partial, bias, rows, slices)
            return out
        with profiler.span("library_gemm"):
            if out_dtype == torch.float32:
                torch.mm(x[:rows], w.t(), out_dtype=torch.float32, out=out[:rows])
                if bias is not None:
                    out[:rows] += bias
            elif bias is not None:
                torch.addmm(bias, x[:rows], w.t(), out=out[:rows])
            else:
                torch.mm(x[:rows], w.t(), out=out[:rows])
        return out

    def _into_residual(self, x, bias, rows, ctx, sink: ResidualSink, used=None):
        """The product added into the residual rows, and the rows of the norm that follows left as
        NormedRows: by the product's own epilogue, or, where it is cut along K, by the kernel
        that adds the slices."""
        N, K = self.weight.shape
        gain, eps, *dyt = sink.norm.carried()
        more = (sink.scale, *dyt) if dyt else (sink.scale,)      # (scale[, Dynamic Tanh's bias, alpha])
        out_pieces = N % 8 == 0
        xg = ctx.alloc(ops.pieces_shape(rows, N) if out_pieces else (rows, N), torch.bfloat16)
        _, a, scale, pieces = _operand(x)
        if rows <= ops.BLOCKSPLIT_PIECES_MAX_M:
            sq = ctx.alloc((rows, ops.gemm_blocksplit_blocks(rows, N, K)), torch.float32)
            ops.gemm_blocksplit(None, a, self.weight, bias, rows, row_scale=scale,
                                residual=(sink.stream.resid, gain, xg, sq, *more), x_pieces=pieces,
                                out_pieces=out_pieces, used=used)
        else:
            groups, splits = self._plan(rows)
            if splits == 1:
                sq = ctx.alloc((rows, groups), torch.float32)
                ops.gemm_rows(None, None, a, self.weight, bias, rows, row_scale=scale,
                              residual=(sink.stream.resid, gain, xg, sq, *more), x_pieces=pieces,
                              out_pieces=out_pieces)
            else:
                partial = ctx.alloc((splits, rows, N), torch.float32)
                ops.gemm_rows(None, partial, a, self.weight, None, rows, row_scale=scale, x_pieces=pieces)
                sq = ctx.alloc((rows, ops.splitk_reduce_residual_blocks(N)), torch.float32)
                ops.splitk_reduce_residual(sink.stream.resid, partial, bias, gain, xg, sq, rows, splits,
                                           out_pieces=out_pieces, scale=sink.scale,
                                           dyt_bias=dyt[0] if dyt else None, dyt_alpha=dyt[1] if dyt else None)
        sink.stream.prepared = (sink.norm, NormedRows(xg, sq, eps, rows, out_pieces, bool(dyt)))
        return None

    def gated_silu_rows(self, rows: int, ctx: StepContext, act: torch.dtype) -> bool:
        """Whether gated_silu applies to this many rows of this dtype."""
        return self._has("gated", rows, ctx, act) and self.weight.shape[0] % 2 == 0

    def gated_silu(self, x, rows: int, ctx: StepContext, out: torch.Tensor,
                   out_pieces: bool = False, act: dict | None = None) -> None:
        """out[rows, N/2] = silu(gate) * up in one kernel, for a weight whose rows alternate gate
        and up (gate i at row 2i, its up at 2i + 1), where gated_silu_rows() says so. x: a tensor,
        NormedRows or PieceRows; out_pieces: out is shaped and written piece-major. act: the
        constants of another gated activation ({alpha, limit, up_shift, cubic} as ops.silu_mul takes them)."""
        act = act or {}
        consts = (act.get("alpha", 1.0), act.get("limit", 0.0), act.get("up_shift", 0.0), act.get("cubic", 0.0))
        act_dtype, a, scale, pieces = _operand(x)
        if not self.gated_silu_rows(rows, ctx, act_dtype):
            raise ValueError("Linear.gated_silu: not for these rows (ask gated_silu_rows)")
        if rows <= ops.BLOCKSPLIT_PIECES_MAX_M:
            ops.gemm_blocksplit(out, a, self.weight, None, rows, gated=True, row_scale=scale,
                                x_pieces=pieces, out_pieces=out_pieces, act=consts, ordered=self.ordered)
            return
        splits = self._plan(rows)[1]
        if splits == 1:
            ops.gemm_rows(out, None, a, self.weight, None, rows, gated=True, row_scale=scale,
                          x_pieces=pieces, out_pieces=out_pieces, act=consts)
            return
        # few weight rows, cut along K: the activation kernel adds the slices while it reads them
        if out_pieces:
            raise ValueError("Linear.gated_silu: a product cut along K writes row-major (ask gated_pieces)")
        partial = ctx.alloc((splits, rows, self.weight.shape[0]), torch.float32)
        ops.gemm_rows(None, partial, a, self.weight, None, rows, row_scale=scale, x_pieces=pieces)
        ops.silu_mul(out, partial, rows, True, splits, **act)

    def _rounds(self, rows: int, bm: int) -> float:
        """The tiles of bm x 256 outputs of this product, in rounds of the chip's units."""
        return -(-rows // bm) * -(-self.weight.shape[0] // 256) / ops.compute_units()

    def tall_gated(self, rows: int, ctx: StepContext, x) -> int:
        """The rows of a tile where the gated product of this many bf16 rows runs as one kernel (kernels.ops.gemm_tall), 0 where it
        is the library's product and an activation kernel. One kernel for K up to 1024 where its tiles are one round on the
        chip: of 128 rows from 0.6 of a round on, of 256 where those are more than a round and 0.7 of the round's outputs are
        real. Over 4879 random weights and row counts that this takes, 0.48 to 1.21 of the time of the two, 0.70 in the geometric mean, 22
        above 1.03, those of some 150 to 320 rows whose second row of tiles is mostly padding (8192 x 1024 at 1000 rows 27.2 us beside 31.6,
        9728 x 896 at 768 rows 22.5 beside 24.9, at 1400 36.4 beside 36.8; 29824 x 704 at 149 rows 1.21). With fewer tiles units idle (1024 x 256 at
        1000 rows 12.7, 8.0)."""
        N, K = self.weight.shape
        if not (K <= 1024 and isinstance(x, torch.Tensor) and x.dtype == BF16 and x.is_contiguous() and K % 64 == 0 and N % 8 == 0
                and ops.tiles_read(x, self.weight) and self.own_tiles(rows, ctx)) or library_tuning.enabled():
            return 0             # (a tuned choice of the library has not been measured against)
        if self._rounds(rows, 128) <= 1:
            return 128 if self._rounds(rows, 128) >= 0.6 else 0
        return 256 if self._rounds(rows, 256) <= 1 and rows * N >= 0.7 * 256 * 256 * ops.compute_units() else 0

    def gated_tile(self, rows: int, ctx: StepContext, x) -> tuple[int, int] | None:
        """The tile (ops.gemm_tall's bm, bn) where a gated product of this many bf16 rows with K above 1024 (up to 1024: tall_gated), or one
        with a relu, runs as one kernel, None where it is the library's product and an activation kernel: one kernel where the tiles of
        gemm_tall_tile's choice are 0.8 of their rounds or more, and either one row of tiles, which read the weight once whatever of
        their rows is padding, or 0.72 of the rounds real outputs. Over 198 gated products of 65 to 12001 rows, 256 to 55296 columns and K up to 20000 it took 0.71 to
        1.09 of the time of the two, 0.90 in the geometric mean, 3 of them above 1.03 (2048 x 37888 x 3584 424 us beside 546, 203 rows 73
        beside 85, 100 rows 58 beside 71); with several rows of tiles and less of them real 0.77 to 1.24 (259 x 28672 x 4096 100 us, the two 82,
        541 x 37888 x 2048 106 and 98), with tiles for less than 0.8 of the rounds up to 1.48. Only where a part allows it (one_round_tiles): see _long."""
        N, K = self.weight.shape
        if not (self.one_round_tiles and K > 1024 and isinstance(x, torch.Tensor) and x.dtype == BF16 and x.is_contiguous() and K % 64 == 0
                and N % 8 == 0 and self.weight.is_contiguous() and ops.tiles_read(x, self.weight) and self.own_tiles(rows, ctx)) \
                or library_tuning.enabled():
            return None
        tile, (tiles, real) = ops.gemm_tall_tile(rows, N, K), self._tile_fill(rows)
        return tile if tiles >= 0.8 and (rows <= tile[0] or real >= 0.72) else None

    def activated(self, x, rows: int, ctx: StepContext, kind: str):
        """unary_act(kind) of the product as one kernel, None where the caller runs the two: up to 16 rows for any kind, many rows
        for the relu ones."""
        act, a, scale, pieces = _operand(x)
        if act != BF16 or not routes.routes_of("linear", (self.weight.dtype, act)):
            return None
        if 0 < rows <= ops.BLOCKSPLIT_PIECES_MAX_M and self.route(rows, ctx, act).run is Linear._run_mfma:
            out = ctx.alloc((rows, self.weight.shape[0]), act)
            ops.gemm_blocksplit(out, a, self.weight, self.bias, rows, row_scale=scale, x_pieces=pieces, unary=kind, ordered=self.ordered)
            return out
        tile = self.gated_tile(rows, ctx, x) if kind in ("relu2", "relu") else None
        if tile is None:
            return None
        out = ctx.alloc((rows, self.weight.shape[0]), act)
        ops.gemm_tall(out, x, self.weight, self.bias, rows, bm=tile[0], bn=tile[1], unary=kind)
        return out

    def gated_pieces(self, rows: int) -> bool:
        """Whether gated_silu can write its result piece-major at this many rows."""
        return rows <= ops.BLOCKSPLIT_PIECES_MAX_M or self._plan(rows)[1] == 1


def _mfma_takes(case: ProductCase) -> bool:
    # the MFMA kernels take K in steps of 8
    return case.fast and case.K % 8 == 0 and 0 < case.rows <= ops.ROWS_MAX_M


routes.register_route("linear", (BF16, BF16), "mfma", _mfma_takes, Linear._run_mfma,
                      traits=("pieces", "gated", "k_slices"))
routes.register_route("linear", (BF16, BF16), "plain", lambda c: not c.fast or c.K % 8 != 0, Linear._run_plain)
routes.register_route("linear", (BF16, BF16), "library", lambda c: True, Linear._run_library)
routes.register_route("linear", (F32, F32), "plain", lambda c: True, Linear._run_plain)
routes.register_route("linear", (F32, BF16), "plain_widened", lambda c: True, Linear._run_plain_widened)
