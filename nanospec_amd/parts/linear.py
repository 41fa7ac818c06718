"""x @ W^T for the parts: ``LinearWeight`` holds a weight matrix and chooses the kernel by precision and row count.

float32: ``csrc/gemm_generic.hip``, 32-bit products and sums in a fixed order: up to 8 rows stream the weights, more run the 32-bit matrix
instruction, odd sizes the plain tiled kernel; and ``csrc/gemm_split.hip`` for many rows, on the float16 matrix cores: each float as the sum of two
float16 values, which stand for it to 2^-23, a product to 2^-21, and sums nearer to 64 bits than the 32-bit instruction's unless nearly
all of a row is zero.  Rows whose values lie too far apart for that, or are infinite, have the 32-bit instruction's results.

bfloat16: decode and short portions (up to ``STREAM_ROWS`` rows) run the hand-written matrix-core kernel that streams
the weights once; it reads them in a layout re-laid at load time (``kernels.ops.TiledWeight``) in which every load
of a wave is one contiguous kilobyte.  17 to 64 rows run a second hand-written kernel on the same layout (x shared
through LDS, K cut into ranges) where it is ahead of the library, and so do products of up to 128 rows that end in the
residual stream (at 65 to 128 rows the library takes two to three times as long for them).  More rows go to the platform's GEMM library on the
plain layout, as the reference's nn.Linear does (model/llama.py:168-171).  32-bit results (logits) always come from the
hand-written kernels, in slices of 64 rows, so that no logit is rounded to bfloat16.  Of the products of more rows those
whose tiles come to about one a compute unit run a third hand-written kernel on the plain layout (``ops.many_plan`` says which).  Both layouts are kept in memory unless
``keep_plain=False``.
"""

from __future__ import annotations

import torch

from ..kernels import ops

# Which copies of a bfloat16 weight matrix a model keeps (``DecoderModel.load(..., layouts=)``; parts that say
# ``takes_layouts`` are told at load time): the re-laid one that the streaming kernels read is always there; the plain one,
# which the library's products for many rows read, only with "both".  With "tiled" many rows run in blocks through the
# hand-written kernels: slower prompts, half the memory.  Of a float32 matrix the plain copy is always there and, with "both", one in
# two parts that its products of many rows read (``ops.SplitWeight``).
LAYOUTS = ("both", "tiled")


STREAM_ROWS = 16  # up to here the streaming kernel beats the library at the shapes measured
GATED_WIDE_ROWS = 80  # up to here gate and up with the activation go through the 17-to-128-row kernel where the library's layout is kept too
WIDE_HEAD_ROWS = 12  # above this many rows a wide 32-bit product (the head) is faster through the 17-to-64-row kernel
WIDE_MAX_N = 4096  # 17 to 64 rows: the hand-written kernel is ahead of the library for outputs up to this width (and for
#                    32-bit results, which the library does not give); wider products go to the library
SPLIT_MIN_K = 8192  # from this inner size on ranges of K are worth a kernel that adds them up, where no norm does it (512 rows of 2,048, K 8,192: 35 / 35
#                     us in the library, alone and beside two others, 32 / 24 in four ranges with that kernel; K 4,096 20 / 15 and 21 / 16)
ACT_FORMS = 3  # the tiles of ``ops.linear_many`` (the first of them) that apply an activation in the product's epilogue: 512 rows of 8,192, K 2,048, in tiles of 128 x 128 30.5 /
#                22.4 us with a kernel behind it and 31.1 / 19.8 in the epilogue, alone and beside two others; the largest tile's epilogue, a workgroup a
#                unit with nothing beside it, costs more than that kernel
LIBRARY_MAX_K = 14336  # the longest inner size over which the library's product has run here, kernel by kernel and inside
#                        captured steps, with every replay checked.  ``library_product`` refuses a longer one: such a product is cut
#                        into slices of its inner size in steps that are launched kernel by kernel, and runs through the
#                        hand-written kernels in captured steps, whichever layouts are kept.
PLAIN_SLICE_K = 8192  # the slices of a product on its way into the residual stream that is cut along its inner size are no
#                       longer than this (where only the re-laid copy is kept the scratch copy is then a slice, not the
#                       matrix, and products are cut from this size on already)
UNTILE_MIN_ROWS = 768  # where only the re-laid copy is kept: from this many rows on the products whose callers allow it
#                        (``plain_copy``: q/k/v, o, gate/up, down) first write their matrices out in plain rows (scratch) and go to
#                        the library; the copy costs what 300 rows of the product cost, and the library is 1.6 to 2 times as
#                        fast as the many-row kernel (measured at the 70B shape).  Callers allow it in steps that are launched
#                        kernel by kernel only: the scratch is as large as the matrix, and every captured step keeps its own.


def library_product(x: torch.Tensor, w_t: torch.Tensor, out: torch.Tensor | None = None, into: torch.Tensor | None = None,
                    plain: torch.Tensor | None = None, take=None, split: bool = False, gated: torch.Tensor | None = None,
                    act: str | None = None):
    """The one door to products of many rows with a matrix in plain rows: x @ w_t (``w_t`` [in, out], usually the transposed view of a
    matrix in plain rows).  ``into``: the product is added to this tensor in place, summed in 32-bit and rounded once; a 32-bit
    ``into`` beside bfloat16 operands keeps the sum in 32-bit.  ``gated`` (with ``plain`` and ``take``): of a product with stacked gate and up matrices
    silu(gate) * up goes there.  ``act``: an activation (``ops.ACTIVATIONS``) of the product (not with ``into``).
    It goes to the platform's GEMM library, or with ``plain`` (``w_t`` untransposed) to ``ops.linear_many`` where that is the faster one (``ops.many_plan``).  ``take`` (shape,
    dtype) gives scratch for ranges of K; with ``split`` (and ``into``) the ranges may come back as a ``PartialSums``, not yet added.
    An inner size beyond ``LIBRARY_MAX_K`` is refused: the library chooses other kernels for it, none of which has run here."""
    m, k = x.shape
    if k > LIBRARY_MAX_K:
        raise ops.KernelRefused(f"a library product over an inner size of {k} (more than {LIBRARY_MAX_K}) must be cut into slices")
    if gated is not None:
        inter = w_t.shape[1] // 2
        plan = ops.many_plan(m, 2 * inter, k, ops.compute_units(x.device), gated=True) if ops.many_takes(x, plain) else None
        if plan is not None and ops.many_writes(gated, m, inter):
            return ops.linear_many(x, plain[:inter], gated, plan[0], w2=plain[inter:])
        return ops.silu_mul(torch.matmul(x, w_t, out=take((m, 2 * inter), x.dtype)), out=gated)
    if plain is not None:
        n, to = w_t.shape[1], into if into is not None else out
        may_split = take is not None and (split if into is not None else k >= SPLIT_MIN_K)
        plan = ops.many_plan(m, n, k, ops.compute_units(x.device), may_split=may_split) if ops.many_takes(x, plain) else None
        if plan is not None and (to is None or ops.many_writes(to, m, n)):
            form, ranges = plan
            if to is None:
                to = torch.empty((m, n), dtype=x.dtype, device=x.device)
            if ranges > 1:
                parts = ops.linear_many(x, plain, take((ranges * m * n,), torch.float32), form, ranges=ranges)
                if into is not None:
                    return parts
                ops.reduce_partial(parts, out=to)
            elif act is not None and form < ACT_FORMS:
                return ops.linear_many(x, plain, to, form, act=act)
            else:
                ops.linear_many(x, plain, to, form, add=into is not None)
            return to if act is None else ops.activation(to, act)
    if into is not None:
        if into.dtype == torch.float32 and x.dtype != torch.float32:
            return torch.addmm(into, x, w_t, out_dtype=torch.float32, out=into)
        return into.addmm_(x, w_t)
    y = torch.matmul(x, w_t) if out is None else torch.matmul(x, w_t, out=out)
    return y if act is None else ops.activation(y, act)


def split_weight(w: torch.Tensor) -> "ops.SplitWeight | None":
    """The second copy of a float32 matrix, for ``product_f32``, or None where that has no use for it."""
    n, k = w.shape
    if w.dtype != torch.float32 or not w.is_cuda or not ops.SPLIT_MIN_K <= k < 1 << 19 or k % ops.SPLIT_K_MULTIPLE or n > 1 << 19 or not ops.split_takes(w[:1], w):
        return None
    return ops.SplitWeight(w)


def product_f32(x: torch.Tensor, w: torch.Tensor, split: "ops.SplitWeight | None", out: torch.Tensor | None, arena) -> torch.Tensor:
    """x @ w^T in 32-bit: many rows of a wide enough matrix on the float16 matrix cores (``ops.linear_split``; its scratch comes from ``arena``, without one it is not taken; ``split``: ``split_weight`` of w), the others on the 32-bit ones."""
    plan = ops.split_plan(x.shape[0], w.shape[0], w.shape[1], ops.compute_units(x.device)) if arena is not None and split is not None else None
    if plan is None or not ops.split_takes(x, w):
        return ops.linear_generic(x, w, out=out)
    mark = arena.mark()
    padded = arena.read_rows is not None and arena.read_rows[0] == x.shape[0]
    out = ops.linear_split(x, w, *plan, out=out, take=arena.take, split=split, read_rows=arena.read_rows[1] if padded else None)
    arena.release(mark)
    return out


def second_copies(part, seen: set | None = None):
    """The weights within ``part`` that keep a second copy of a float32 matrix (``split_weight``)."""
    seen = set() if seen is None else seen
    if id(part) in seen:
        return
    seen.add(id(part))
    if isinstance(part, (LinearWeight, GatedWeights)) and part._split is not None:
        yield part
    inside = part if isinstance(part, (list, tuple)) else part.values() if isinstance(part, dict) else vars(part).values() if type(part).__module__.startswith(__package__) else ()
    for one in inside:
        yield from second_copies(one, seen)


SPLIT_MOST_LOST = 0.125  # of the rows of a matrix, by 16, whose values may lie too far apart for the parts


def drop_copies_of_little_use(part) -> None:
    """Second copies within ``part`` that do not stand for too many of the matrix's rows are let go: each 16 such rows are made by the 32-bit instruction behind every product, which is slower than the 32-bit
    product of all alone where they are many.  us, that product and the split one with none, an eighth and a quarter of them so: 832 rows, N = K = 2,048 62 and 45, 68, 67, N 2,048, K 8,192 244 and 123, 217, 225, N 16,384, K 2,048
    546 and 204, 302, 376; 128 rows of the last 68 and 41, 66, 67.  (One trip to the GPU for all of them: a matrix by itself as it is split costs a model of 32 matrices a millisecond of its load.)"""
    holders = list(second_copies(part))
    if holders:
        for holder, lost in zip(holders, torch.stack([h._split.lost[0] for h in holders]).tolist()):
            if lost > SPLIT_MOST_LOST * -(-holder._split.n // 16):
                holder._split = None


class IntoResidual:
    """Asks a part to hand its output to the residual stream and the RMS norm after it in the cheapest form its last
    product has, instead of returning a finished tensor:
      * ``kernels.ops.PreNormed``: ``resid += output`` has been done in place and the norm needs no kernel of its own
        (at most 16 rows: the product's epilogue did the sum and the norm's statistics);
      * ``kernels.ops.PartialSums``: the ranges of a product whose K was cut, which the norm kernel adds up as it reads
        them (17 to 128 rows, and more where their tiles alone leave most of the GPU idle);
      * ``kernels.ops.Added``: ``resid += output`` has been done in place by the product itself (more rows),
        the norm still has its kernel;
      * a tensor: the output, still to be added by the norm kernel.
    ``next_weight``, ``eps``: that norm's weight and epsilon.  ``x_next`` (like resid), ``ssq`` (float32 [rows,
    ceil(width / 16)]) and ``carry`` (float32, room for the ranges: 16 * rows * width for up to 128 rows, ``ops.many_ranges`` for more): where the results go if they must outlive the block's
    scratch (``outlives``); otherwise scratch is taken."""

    def __init__(self, resid: torch.Tensor, next_weight: torch.Tensor, eps: float, x_next: torch.Tensor | None = None,
                 ssq: torch.Tensor | None = None, carry: torch.Tensor | None = None, outlives: bool = False) -> None:
        self.resid, self.next_weight, self.eps = resid, next_weight, eps
        self.x_next, self.ssq, self.carry, self.outlives = x_next, ssq, carry, outlives


class LinearWeight:
    def __init__(self, w: torch.Tensor, keep_plain: bool = True, tiled: bool = True) -> None:
        """``w``: [out, in] on the GPU in the compute dtype.  ``tiled=False``: the caller streams this matrix with a
        kernel and a layout of its own for few rows, so only the plain layout is kept here.  ``keep_plain=False``: only the
        re-laid copy is kept (see ``LAYOUTS``)."""
        self.n, self.k = w.shape
        self.dtype = w.dtype
        fast = w.dtype == torch.bfloat16 and self.k % 8 == 0
        # (an inner size that the library does not take in one piece needs the hand-written kernels for many rows too)
        self.tiled = ops.TiledWeight(w) if (fast and (tiled or self.k > LIBRARY_MAX_K)) else None
        self.plain = w if (keep_plain or self.tiled is None) else None
        self._plain_t = self.plain.t() if self.plain is not None else None  # the library product's operand, made once
        self._split = split_weight(w) if keep_plain else None

    def links_norms(self, rows: int) -> bool:
        """Whether a product of ``rows`` rows can take a ``PreNormed`` input and can end in the residual stream."""
        return self.tiled is not None and rows <= STREAM_ROWS

    def into_residual(self, x: torch.Tensor, link: IntoResidual, arena=None, plain_copy: bool = False):
        """x @ W^T on its way into the residual stream, in one of the forms ``IntoResidual`` names.  ``plain_copy``: as for
        ``__call__``."""
        m = x.shape[0]
        take = (lambda shape, dtype: arena.take(shape, dtype)) if arena is not None else (lambda shape, dtype: torch.empty(shape, dtype=dtype, device=x.device))
        if self.links_norms(m) and x.dtype == torch.bfloat16 and ops.tiled_takes(x[:1], self.k):
            x_next = link.x_next if link.x_next is not None else take(tuple(link.resid.shape), link.resid.dtype)
            ssq = link.ssq if link.ssq is not None else take((m, -(-self.n // 16)), torch.float32)
            return ops.linear_resid_norm(x, self.tiled, link.resid, link.next_weight, link.eps, x_next=x_next, ssq=ssq)
        if (self.tiled is not None and STREAM_ROWS < m <= ops.WIDE_TALL_ROWS and (self.plain is None or self.n <= WIDE_MAX_N)
                and x.dtype == torch.bfloat16 and ops.tiled_takes(x[:1], self.k)):
            ksplit, nt = ops.wide_plan(self.n, self.k, m)
            need = ksplit * m * self.n
            ws = None
            if ksplit > 1 and link.carry is not None and link.carry.numel() >= need:
                ws = link.carry
            elif ksplit > 1 and not link.outlives:
                ws = take((need,), torch.float32)
            if ws is not None:
                return ops.linear_wide(x, self.tiled, workspace=ws, ksplit=ksplit, nt=nt, defer=True)
        r = link.resid
        # many rows: the library's product takes the stream as its addend, resid = resid + x @ W^T summed in 32-bit and
        # rounded once, so the norm after it reads one tensor instead of two and writes one instead of two
        library = (m > ops.SKINNY_MAX_ROWS and x.dtype == torch.bfloat16 and r.dtype == torch.bfloat16 and r.shape == (m, self.n)
                   and r.is_contiguous())
        have_plain = self._plain_t is not None
        # only the re-laid copy is kept: many rows of a step that is launched kernel by kernel may copy it into plain rows
        can_copy = (not have_plain and plain_copy and self.tiled is not None and m >= UNTILE_MIN_ROWS and ops.tiled_takes(x[:1], self.k))
        if library and (have_plain or can_copy):
            if self.k > (LIBRARY_MAX_K if have_plain else PLAIN_SLICE_K):
                if plain_copy:
                    # a long inner size in slices: the stream in 32-bit takes every slice's product as the library adds it
                    # (32-bit sums, 32-bit addend and result) and is rounded once at the end, as one product would be
                    slices = -(-self.k // PLAIN_SLICE_K)
                    width = -(-self.k // (128 * slices)) * 128
                    acc = take((m, self.n), torch.float32)
                    acc.copy_(r)
                    scratch = None if have_plain else take((self.n, width), self.dtype)
                    for k0 in range(0, self.k, width):
                        k1 = min(self.k, k0 + width)
                        piece = self.plain[:, k0:k1] if have_plain else ops.untile(self.tiled, scratch[:, : k1 - k0], k0, k1)
                        library_product(x[:, k0:k1], piece.t(), into=acc)
                    r.copy_(acc)
                    return ops.Added()
                # (a captured step: the hand-written kernels below)
            else:
                if not have_plain:
                    library_product(x, ops.untile(self.tiled, take((self.n, self.k), self.dtype)).t(), into=r)
                    return ops.Added()
                # (ranges of K, where the product is cut, lie where the norm still finds them)
                room = (lambda shape, dtype: link.carry) if link.carry is not None else take
                split = (not link.outlives if link.carry is None
                         else link.carry.numel() >= ops.many_ranges(m, self.n, ops.compute_units(x.device)) * m * self.n)
                done = library_product(x, self._plain_t, into=r, plain=self.plain, take=room, split=split)
                return done if isinstance(done, ops.PartialSums) else ops.Added()
        out = link.x_next if link.x_next is not None else take((m, self.n), x.dtype)
        return self(x, out=out, arena=arena, plain_copy=plain_copy)

    def __call__(self, x, out: torch.Tensor | None = None, out_f32: bool = False, arena=None, plain_copy: bool = False,
                 act: str | None = None) -> torch.Tensor:
        """``arena``: where the workspace of the 17-to-64-row kernel comes from (``ctx.arena``); without it it is allocated.
        ``x`` may be a ``PreNormed`` where ``links_norms`` holds.  ``plain_copy``: where only the re-laid copy is kept, many
        rows may go to the library through a plain copy of the matrix in scratch (see ``UNTILE_MIN_ROWS``).  ``act``: an
        activation (``ops.ACTIVATIONS``) on the result: in the product's epilogue for few rows and for many where it is the
        faster one, a kernel of its own otherwise; the values are the same either way."""
        if act is not None:
            if (not out_f32 and self.tiled is not None and not isinstance(x, ops.PreNormed) and x.shape[0] <= STREAM_ROWS
                    and x.dtype == self.dtype and ops.tiled_takes(x[:1], self.k)):
                return ops.linear_tiled(x, self.tiled, out=out, act=act)
            if (not out_f32 and self.plain is not None and x.dtype == self.dtype and x.shape[0] >= ops.MANY_MIN_ROWS and self.k <= LIBRARY_MAX_K
                    and ops.many_takes(x, self.plain)):
                scratch = arena.take if arena is not None else (lambda shape, dtype: torch.empty(shape, dtype=dtype, device=x.device))
                return library_product(x, self._plain_t, out=out, plain=self.plain, take=scratch, act=act)
            return ops.activation(self(x, out=out, out_f32=out_f32, arena=arena, plain_copy=plain_copy), act)
        if isinstance(x, ops.PreNormed):
            if not self.links_norms(x.shape[0]):
                raise ops.KernelRefused("this product cannot take a pre-normed input (rows, layout or precision)")
            return ops.linear_tiled(x, self.tiled, out=out, out_f32=out_f32)
        if x.dtype != self.dtype:
            raise ops.KernelRefused(f"linear: input is {x.dtype}, the weight {self.dtype}")
        if self.dtype == torch.float32:
            return product_f32(x, self.plain, self._split, out, arena)
        if self.k % 8 or not ops.tiled_takes(x[:1], self.k):
            return ops.linear_generic(x, self.plain, out=out, out_f32=out_f32)
        m = x.shape[0]
        ranges = None
        if (out_f32 and m >= ops.MANY_MIN_ROWS and self.plain is not None and ops.many_f32_takes(x, self.plain)
                and (out is None or out.dtype == torch.float32 and out.is_contiguous() and out.data_ptr() % 16 == 0)):
            ranges = ops.many_f32_ranges(m, self.n, self.k, ops.compute_units(x.device))
        if ranges is not None:
            # (us in blocks of 128 rows from the re-laid copy and here, alone / beside two others: 2,048 columns, K 4,096, 130 rows 28.8 / 24.8, 15.3 / 9.7, 508 37.7 / 30.8, 21.1 / 15.5, 2,048 71 / 66,
            # 46 / 42; 4,096 columns, K 8,192, 508 rows 69 / 64, 44 / 40, 2,048 203 / 205, 114 / 117.  Both 1.9e-7 to 5.7e-7 from 64 bits, the same of either; in one range 35 / 34 in the third of these, but
            # 4.0e-7 for 2.7e-7)
            if out is None:
                out = torch.empty((m, self.n), dtype=torch.float32, device=x.device)
            if ranges == 1:
                return ops.linear_many(x, self.plain, out, ops.MANY_SPLIT_FORM)
            sums = arena.take((ranges * m * self.n,), torch.float32) if arena is not None else torch.empty(ranges * m * self.n, dtype=torch.float32, device=x.device)
            return ops.reduce_partial(ops.linear_many(x, self.plain, sums, ops.MANY_SPLIT_FORM, ranges=ranges), out=out)
        if self.tiled is not None and WIDE_HEAD_ROWS < m <= STREAM_ROWS and out_f32 and self.n >= 8192:
            return ops.linear_wide(x, self.tiled, out=out, out_f32=True, ksplit=1, nt=1)
        if self.tiled is not None and m <= STREAM_ROWS:
            return ops.linear_tiled(x, self.tiled, out=out, out_f32=out_f32)
        if self.tiled is not None and m <= ops.SKINNY_MAX_ROWS and (out_f32 or self.plain is None or self.n <= WIDE_MAX_N):
            ksplit, nt = ops.wide_plan(self.n, self.k)
            ws = arena.take((ksplit * m * self.n,), torch.float32) if (arena is not None and ksplit > 1) else None
            return ops.linear_wide(x, self.tiled, out=out, out_f32=out_f32, workspace=ws, ksplit=ksplit, nt=nt)
        if self.tiled is not None and m <= ops.WIDE_TALL_ROWS and self.n <= WIDE_MAX_N:
            # 65 to 128 rows of a narrow product (the last layer's down-projection, which no norm inside the layer loop follows)
            ksplit, nt = ops.wide_plan(self.n, self.k, m)
            ws = arena.take((ksplit * m * self.n,), torch.float32) if (arena is not None and ksplit > 1) else None
            return ops.linear_wide(x, self.tiled, out=out, out_f32=out_f32, workspace=ws, ksplit=ksplit, nt=nt)
        if self.plain is not None and (not out_f32 or self.tiled is None) and (self.k <= LIBRARY_MAX_K or self.tiled is None):
            if out_f32:
                return ops.linear_generic(x, self.plain, out=out, out_f32=True)
            scratch = arena.take if arena is not None else (lambda shape, dtype: torch.empty(shape, dtype=dtype, device=x.device))
            return library_product(x, self._plain_t, out=out, plain=self.plain, take=scratch)
        if out is None:
            out = torch.empty((m, self.n), dtype=torch.float32 if out_f32 else x.dtype, device=x.device)
        if self.plain is None and m >= UNTILE_MIN_ROWS and not out_f32 and plain_copy and self.k <= PLAIN_SLICE_K:  # only the tiled layout is kept, many rows: a plain copy for this one product
            plain = arena.take((self.n, self.k), self.dtype) if arena is not None else torch.empty((self.n, self.k), dtype=self.dtype, device=x.device)
            return library_product(x, ops.untile(self.tiled, plain).t(), out=out)
        if m > ops.WIDE_TALL_ROWS:  # ... fewer: blocks of 128 rows through the hand-written kernel
            ksplit, nt = ops.rows_plan(self.n, self.k, m)
            ws = arena.take((ksplit * m * self.n,), torch.float32) if (arena is not None and ksplit > 1) else None
            return ops.linear_rows(x, self.tiled, out=out, out_f32=out_f32, workspace=ws, ksplit=ksplit, nt=nt)
        ksplit, nt = ops.wide_plan(self.n, self.k)
        ws = arena.take((ksplit * ops.SKINNY_MAX_ROWS * self.n,), torch.float32) if (arena is not None and ksplit > 1) else None
        for s in range(0, m, ops.SKINNY_MAX_ROWS):
            e = min(m, s + ops.SKINNY_MAX_ROWS)
            if e - s <= STREAM_ROWS:
                ops.linear_tiled(x[s:e], self.tiled, out=out[s:e], out_f32=out_f32)
            else:
                ops.linear_wide(x[s:e], self.tiled, out=out[s:e], out_f32=out_f32, workspace=ws, ksplit=ksplit, nt=nt)
        return out


class GatedWeights:
    """Gate and up matrices of a gated feed-forward: silu(x @ Wg^T) * (x @ Wu^T) in one pass over x.  ``bias`` = (gate's,
    up's): silu(x @ Wg^T + bg) * (x @ Wu^T + bu); up to 16 rows add them in the streaming product's epilogue, more rows go
    through the product of the stacked matrices and a kernel that adds the biases and applies the activation."""

    def __init__(self, gate: torch.Tensor, up: torch.Tensor, keep_plain: bool = True, bias: tuple | None = None) -> None:
        self.inter, self.k = gate.shape
        self.dtype = gate.dtype
        fast = gate.dtype == torch.bfloat16 and self.k % 8 == 0
        self.tiled = (ops.TiledWeight(gate), ops.TiledWeight(up)) if fast else None
        self.bias = None if bias is None else (bias[0].contiguous(), bias[1].contiguous())
        self.bias_stacked = None if bias is None else torch.cat(self.bias).contiguous()
        # [2 I, K] for the two-kernel path (which biased products of more than 16 rows always take)
        self.stacked = torch.cat([gate, up]) if (keep_plain or not fast or bias is not None) else None
        self._stacked_t = self.stacked.t() if self.stacked is not None else None
        self._split = split_weight(self.stacked) if self.stacked is not None and keep_plain else None
        # biased and bfloat16: more than 16 rows take the stacked matrix in plain rows to the library (no third copy is re-laid)
        self._stacked_linear = LinearWeight(self.stacked, keep_plain=True, tiled=False) if (bias is not None and fast) else None

    def links_norms(self, rows: int) -> bool:
        return self.bias is None and self.tiled is not None and rows <= STREAM_ROWS

    def _few_rows(self, x, m: int, out: torch.Tensor) -> torch.Tensor:
        """Up to 16 rows (plain or pre-normed).  From a few rows on, where the number of row tiles deals unevenly to the
        compute units as whole tiles, the kernel that shares x through LDS and takes half tiles is ahead of the one that
        streams a tile per workgroup (8B shape, 896 tiles on 256 units: 37.6 against 39.7 us at 8 rows, 37.4 against 43.8
        at 16); where the tiles deal evenly it is not (1B shape, 512 tiles: 2% of a decode step behind)."""
        tiles, units = -(-self.inter // 16), ops.compute_units(out.device)
        uneven = -(-tiles // units) * units > 1.05 * tiles  # a tile of each matrix per workgroup leaves some units a round short
        if self.bias is not None:
            return ops.linear_tiled(x, self.tiled[0], w2=self.tiled[1], out=out, bias=self.bias[0], bias2=self.bias[1])
        if m > ops.GATED_HALF_ROWS and uneven and ops.wide_waves(self.inter, self.k, m, 1, 1, gated=True, units=units)[1]:
            return ops.linear_wide(x, self.tiled[0], w2=self.tiled[1], out=out, ksplit=1, nt=1)
        return ops.linear_tiled(x, self.tiled[0], w2=self.tiled[1], out=out)

    def __call__(self, ctx, x, out: torch.Tensor) -> torch.Tensor:
        m = x.shape[0]
        if isinstance(x, ops.PreNormed):
            if not self.links_norms(m):
                raise ops.KernelRefused("this product cannot take a pre-normed input (rows, layout or precision)")
            return self._few_rows(x, m, out)
        fast = self.tiled is not None and ops.tiled_takes(x[:1], self.k)
        if fast and m <= STREAM_ROWS:
            return self._few_rows(x, m, out)
        if self.bias is not None:
            gu = ctx.arena.take((m, 2 * self.inter), x.dtype)
            if self._stacked_linear is not None:
                self._stacked_linear(x, out=gu, arena=ctx.arena, plain_copy=not ctx.captured)
            elif self.dtype == torch.float32:
                product_f32(x, self.stacked, self._split, gu, ctx.arena)
            else:
                ops.linear_generic(x, self.stacked, out=gu)
            return ops.silu_mul_bias(gu, self.bias_stacked, out=out)
        # (an inner size that the library does not take in one piece: the hand-written kernels at every number of rows)
        stacked = self.stacked if (self.k <= LIBRARY_MAX_K or not fast) else None
        if fast and stacked is None and self.k <= LIBRARY_MAX_K and m >= UNTILE_MIN_ROWS and not ctx.captured:
            # only the tiled layout is kept, many rows: both matrices in plain rows into scratch, then as with both layouts
            # (not in a captured step: every captured shape would hold a scratch of its own as large as the two matrices)
            stacked = ctx.arena.take((2 * self.inter, self.k), x.dtype)
            ops.untile(self.tiled[0], stacked[: self.inter])
            ops.untile(self.tiled[1], stacked[self.inter :])
            gu = ctx.arena.take((m, 2 * self.inter), x.dtype)
            library_product(x, stacked.t(), out=gu)
            return ops.silu_mul(gu, out=out)
        if fast and stacked is None and m > ops.WIDE_TALL_ROWS:
            # only the tiled layout is kept: blocks of 128 rows through the hand-written kernel, activation in the same pass
            return ops.linear_rows(x, self.tiled[0], w2=self.tiled[1], out=out, ksplit=1, nt=2)
        if fast and (m <= GATED_WIDE_ROWS or stacked is None):
            # 17 to 80 rows: the second hand-written kernel, one range of K, so that the activation is applied in the same
            # pass (measured ahead of the library's product plus the activation kernel: 50 against 60 us at 72 rows of the
            # 8B shape, level at 96).  Beyond 64 rows it holds the sums of both matrices only by half tiles; where only the
            # tiled layout is kept it takes up to 128 rows a pass that way (70B shape: 243 us where two passes of 64 take 331).
            step = ops.WIDE_TALL_ROWS if ops.wide_waves(self.inter, self.k, ops.WIDE_TALL_ROWS, 1, 1, gated=True)[1] else ops.SKINNY_MAX_ROWS
            for s in range(0, m, step):
                e = min(m, s + step)
                ops.linear_wide(x[s:e], self.tiled[0], w2=self.tiled[1], out=out[s:e], ksplit=1, nt=1)
            return out
        if self.dtype == torch.float32 or self.k % 8:
            gu = ctx.arena.take((m, 2 * self.inter), x.dtype)
            product = product_f32(x, self.stacked, self._split, gu, ctx.arena) if self.dtype == torch.float32 else ops.linear_generic(x, self.stacked, out=gu)
            return ops.silu_mul(product, out=out)
        return library_product(x, self._stacked_t, gated=out, plain=self.stacked, take=ctx.arena.take)
