"""Chooses the matrix-product kernel for a linear layer, and carries a LayerNorm that has not
been computed yet to the kernel that can compute it in its prologue."""

from __future__ import annotations

from typing import Optional, Union

import torch

from . import kernels, residual


class LazyNorm:
    """The normed residual stream, not yet computed: norm(x[rows]) (or norm(x)).  A linear layer
    that reads it may compute the norm in its own prologue; anyone else calls tensor()."""

    def __init__(self, norm, x: torch.Tensor, n_rows: int, rows: Optional[torch.Tensor] = None,
                 buffer: str = "normed") -> None:
        self.norm, self.x, self.n_rows, self.rows, self.buffer = norm, x, n_rows, rows, buffer
        self._tensor: Optional[torch.Tensor] = None

    def tensor(self, ctx) -> torch.Tensor:
        if self._tensor is None:
            h = ctx.workspace.get(self.buffer, self.n_rows, self.x.shape[1], ctx.dtype)
            pending = getattr(ctx, "pending", None)
            if pending is not None:
                # the residual is still a sum: a LayerNorm adds it up on its way in (and, where it
                # goes over all the step's rows, stores the sums: the residual is plain again),
                # anything else needs plain rows first
                norm = self.norm
                all_rows = self.rows is None and self.n_rows >= ctx.n_rows
                if (getattr(norm, "fusable_layer_norm", False)
                        and kernels.residual_layer_norm(pending, norm.weight, norm.bias, norm.eps, self.rows, h,
                                                        self.n_rows, settled=self.x if all_rows else None)):
                    if all_rows:
                        ctx.pending = None
                else:
                    residual.settle(ctx, self.x, ctx.n_rows)
                    pending = None
            if pending is None:
                self.norm.forward(ctx, self.x, h, self.n_rows, rows=self.rows)
            self._tensor = h
        return self._tensor


# Derived copies of a matrix (folded with a LayerNorm, packed for the decode kernel) hang on the
# matrix tensor itself, so they live exactly as long as it does.
_DERIVED = "_mgpt_derived"


def _derived(w: torch.Tensor) -> dict:
    """The table of w's derived copies.  It hangs on the tensor that owns the memory (a view made
    afresh at every call would take its table with it when it goes), one table per place and shape."""
    owner = w._base if w._base is not None else w
    tables = getattr(owner, _DERIVED, None)
    if tables is None:
        tables = {}
        setattr(owner, _DERIVED, tables)
    return tables.setdefault((w.data_ptr(), tuple(w.shape), tuple(w.stride())), {})


def derived_bytes(w: torch.Tensor) -> int:
    """Bytes of device memory that the derived copies of w hold (folded with a LayerNorm, packed
    for the decode kernels), counting every copy of every view of w's storage once."""
    owner = w._base if w._base is not None else w
    seen, total = set(), 0

    def walk(obj) -> None:
        nonlocal total
        if isinstance(obj, torch.Tensor):
            if obj.data_ptr() not in seen:
                seen.add(obj.data_ptr())
                total += obj.numel() * obj.element_size()
        elif isinstance(obj, (tuple, list)):
            for item in obj:
                walk(item)
        elif isinstance(obj, dict):
            for item in obj.values():
                walk(item)

    walk(getattr(owner, _DERIVED, None))
    return total


class CopyBudget:
    """Device memory that derived copies of matrices may still take (EngineConfig.derived_weight_bytes).
    A copy that does not fit is not made: its matrix is then read as it was loaded (row-major through
    the decode kernels, its LayerNorm by the LayerNorm kernel), slower and with the same results up
    to rounding."""

    def __init__(self, limit: Optional[int]) -> None:
        self.limit = limit          # None: no bound
        self.used = 0

    def take(self, n_bytes: int) -> bool:
        if self.limit is not None and self.used + n_bytes > self.limit:
            return False
        self.used += n_bytes
        return True


def _budget(ctx) -> Optional[CopyBudget]:
    return getattr(ctx, "copy_budget", None) if ctx is not None else None


def folded_layer_norm(norm, w: torch.Tensor, bias: Optional[torch.Tensor], ctx=None):
    """(folded matrix, column sums, folded bias): the matrix with the LayerNorm's gain and bias
    folded in, made once per (norm, matrix, bias).  None if the step's budget for copies has no
    room for it."""
    key = ("folded", norm.weight.data_ptr(), 0 if norm.bias is None else norm.bias.data_ptr(),
           0 if bias is None else bias.data_ptr())
    d = _derived(w)
    hit = d.get(key)
    if hit is None:
        budget = _budget(ctx)
        if budget is not None and not budget.take(w.numel() * w.element_size() + 8 * w.shape[0]):
            return None
        hit = d[key] = kernels.fold_layer_norm(w, norm.weight, norm.bias, bias)
    return hit


def packed_weight(w: torch.Tensor, ctx=None) -> Optional[torch.Tensor]:
    """The matrix in the layout the decode kernel reads fastest, made once per matrix (at its first
    decode step, before any graph is captured).  None if the kernel's layout does not take the
    shape, or if the step's budget for copies has no room for it."""
    d = _derived(w)
    if "packed" not in d:
        budget = _budget(ctx)
        if budget is not None and w.shape[1] % 32 == 0 \
                and not budget.take(-(-w.shape[0] // 16) * 16 * w.shape[1] * w.element_size()):
            return None         # (not remembered: a later step never has more room, but a test may lift the bound)
        d["packed"] = kernels.pack_weight(w)
    return d["packed"]


# A LayerNorm is folded into the product that reads it only for outputs this wide at most, and for
# this many rows unless the decode kernel deals the rows out in groups of 16: every workgroup
# converts the float32 residual rows it multiplies, which beyond these costs more than a LayerNorm
# kernel of its own (at 64 rows in one workgroup the decode step of the 50.9M model took 0.397 ms
# with the fold and 0.375 ms without).
FOLD_MAX_ROWS = 32
FOLD_MAX_OUT = 4096
# ... except at few rows, where the LayerNorm kernel's own launch costs more than the conversion
# (the GPT-2-XL shape, outputs of 4800 and 6400: 957 us a step of 24 layers against 1062 at one
# row, 1361 against 1399 at 16 rows, 1923 against 1741 at 32), but not under an output as wide as a
# vocabulary: every one of its thousands of workgroups would norm the rows again ([50257 x 1600] at
# one row: 43.5 us with the fold, 30.0 without, and the LayerNorm kernel takes 3)
FOLD_ANY_OUT_MAX_ROWS = 16
FOLD_ANY_OUT_MAX_OUT = 8192
# A very wide output (the head, 8192 columns and more) goes to the decode kernel while rows x inner
# size stays within this, and to the tiled kernel beyond: that one streams the matrix at nearly the
# same rate whatever the rows (50304 x 512: 10.2 us at 1 row, 11.4 at 32, 14.0 at 64), the decode
# kernel is ahead by up to a microsecond at few rows and a short inner size and slows down with every
# row (9.4, 16.4, 28.5 us; at an inner size of 1600 it is behind from 4 rows on).
WIDE_OUT = 8192
WIDE_OUT_DECODE_WORK = 8192


def wide_rows_once(n_rows: int, n_out: int, k_dim: int) -> bool:
    """Whether a very wide output beyond that work goes to the kernel that reads the matrix once, whole lines a load, for a tile of 16 rows
    (linear_rows_once).  Its time grows with the rows, from a lower level than the tiled kernel's where rows of 4,096 bytes and multiples
    come to that one from few of the memory's channels at a time, and does not jump with the rounds of its tiles (at 8,193 and 10,753
    columns, less under an inner size of 2,048).  Tiled / here, us: 32768 x 2048 33.8 / 28.7 at 8 rows, 33.9 / 29.8 at 12, 50257 x 2048 44.5 /
    43.1 and 45.4 / 45.1, 14336 x 2048 14.4 / 13.9 at 5, 14.6 / 14.5 at 12 (8192 x 2048 9.1 / 9.9, 13000 x 2048 12.9 / 13.3 at 5); 8192 x 4096
    18.6 / 16.2 at 3, 18.7 / 16.4 at 12, 32768 x 4096 63.5 / 51.5, 63.9 / 56.1; 12288 x 6144 38.7 / 32.8 at 2, 38.9 / 32.7 at 8, 13000 x 6144
    39.5 / 40.0 at 10; 16384 x 8192 57 / 57 at 3 and 12; 14336 x 10240 63.8 / 63.6 at 6, 64.5 / 65.8 at 8; in between, 9216 x 4096 19.6 / 18.6 at
    3, 20.1 / 21.2 at 12, 9216 x 6144 27.4 / 26.9 at 3, 27.6 / 28.6 at 6."""
    if k_dim % 2048 or (k_dim == 2048 and n_out < 14336):
        return False
    if k_dim > 2048 and 8192 < n_out < 11264:
        return n_rows * k_dim <= 20000
    return n_rows <= (12 if k_dim <= 4096 or k_dim == 8192 else 8 if k_dim < 8192 else 6)


# The decode kernel's time grows with the rows (every workgroup loads all of them for its 16 output
# columns), the tiled kernel's hardly: under a large matrix with a wide output the tiled kernel (32 x
# 32 tiles, several steps on their way from memory) is ahead from 17 rows on.  Matrices from memory,
# decode kernel against tiled: [4800 x 1600] 8.5 / 8.5 us at 16 rows, 10.6 / 8.5 at 24, 11.7 / 8.5 at
# 32, 18.8 / 10.0 at 64; [6400 x 1600] 9.3 / 9.1, 11.4 / 9.3, 12.7 / 9.3, 19.8 / 12.0; under smaller
# matrices the decode kernel stays ahead up to 64 rows ([3072 x 768] 5.0 / 5.6 at 32, 6.2 / 5.6 at
# 64; [1600 x 1600] 5.8 / 8.4 and 8.0 / 8.4).
TILED_FROM_ROWS = 17
TILED_MIN_OUT = 4096
TILED_MIN_MATRIX = 6_000_000
TILED_ANY_SHAPE_FROM_ROWS = 33
# A long inner size under a narrow output is split over workgroups by the tiled kernel, and by the decode kernel where its four
# stretches are whole and the output has fewer than 128 column tiles.  Lines (rows) where the sums are left pending for a LayerNorm,
# and where a second kernel adds them up.  us with the LayerNorm, decode kernel / tiled:
# - where the decode kernel splits: pending [1600 x 6400] 11.5 / 11.0 at 9 rows, 16.3 / 11.3 at 32, [1152 x 4608] 10.6 / 10.3, 15.7 /
#   10.6; added up [1600 x 6400] 13.9 / 14.0 at 16, 14.6 / 13.7 at 17, 17.5 / 13.8 at 32.
# - outputs of 1,024 and less, whose tiles are few: pending [1024 x 8192] 10.1 / 10.8 at 16, 11.0 / 10.8 at 17; added up 11.7 / 12.7 at
#   17, 12.5 / 13.1 at 32.
# - where the decode kernel does not split and the tiled one's slices go straight into LDS: pending [2048 x 4160] 11.7 / 10.8 at 9,
#   15.3 / 11.5 at 32; added up 13.3 / 14.1 at 17, 14.5 / 14.5 at 28, [2048 x 8192] 19.0 / 18.6 at 17, [2560 x 10240] 24.5 / 25.5 at 17,
#   26.8 / 26.3 at 28, [2560 x 5120] 17.1 / 17.7 at 32.
# - through registers (no whole steps of 64): pending [1216 x 4128] 9.8 / 10.5 at 9, 10.5 / 10.6 at 16; added up 12.0 / 13.1 at 32,
#   [1344 x 4128] 14.1 / 14.5 at 40, 15.1 / 14.8 at 48.
TILED_LONG_MIN_INNER = 4097
TILED_LONG_MIN_MATRIX = 5_000_000


def _long_inner_lines(n_out: int, k_dim: int):
    """(rows from which on the sums are left pending, rows from which on they are added up) by the tiled kernel."""
    if n_out <= 1024:
        return 17, 33
    if kernels.linear_skinny_partials(17, n_out, k_dim, False, kernels.EPI_RESIDUAL):
        return 9, 17
    if k_dim % 64:
        return 17, 33 if n_out * k_dim >= TILED_MIN_MATRIX else 41
    return 9, 28 if n_out <= 2048 or k_dim >= 5632 else 33


def tiled_at_few_rows(n_rows: int, w: torch.Tensor, left: bool = False) -> bool:
    """Whether a product of few rows (the decode kernel takes up to 64; linear_add asks for up to
    LEAVE_PARTS_MAX_ROWS) goes to the tiled kernel rather than the decode kernel.  left: the sums of a split
    product are left pending."""
    n_out, k_dim = w.shape
    if n_rows > 8 and n_out < TILED_MIN_OUT and k_dim >= TILED_LONG_MIN_INNER and n_out * k_dim >= TILED_LONG_MIN_MATRIX:
        return n_rows >= _long_inner_lines(n_out, k_dim)[0 if left else 1]
    if n_out * k_dim < TILED_MIN_MATRIX:
        return False
    return n_rows >= TILED_ANY_SHAPE_FROM_ROWS or (n_rows >= TILED_FROM_ROWS and n_out >= TILED_MIN_OUT)


def folds_before_rows_apart(n_rows: int, n_out: int, k_dim: int) -> bool:
    """Whether the LayerNorm of a product that has a kernels.linear_rows_plan is folded into the decode kernel instead.  The fold's work
    grows with the rows in every workgroup (in steps of 8 rows, of 4 beyond an inner size of 2,048); a LayerNorm of its own is a launch of
    2 us, and one of more than 4,096 columns takes ten times that.  Folded / LayerNorm and product, us: 768 -> 2304 3.3 / 4.8 at 1 row, 5.0 /
    5.2 at 16, 6.4 / 5.5 at 24; 1024 -> 4096 6.0 / 6.3 at 16, 8.3 / 6.7 at 24; 960 -> 1792 5.3 / 5.9 at 32; short inner sizes always (512 ->
    1536 3.9 / 5.5 at 32).  1280 -> 3840 6.6 / 7.0 at 8, 7.9 / 7.1 at 12; 2048 -> 3072 7.3 / 8.0 at 8, 8.4 / 8.2 at 12; 3072 -> 2048 8.1 / 8.4
    at 4, 9.3 / 8.7 at 6.  While workgroups of 8 rows and 16 columns all have a compute unit, under small matrices: 1600 -> 1024 5.5 / 6.9 at
    32, 1408 -> 1280 5.4 / 6.5 at 24 and 7.2 / 6.5 at 28, 1600 -> 1792 5.8 / 6.4 at 16 (1792 -> 1792 8.0 / 6.4).  With more than a workgroup
    of 16 columns a compute unit: 1280 -> 5120 7.4 / 7.6 at 4, 8.5 / 7.9 at 8, 12.6 / 8.3 at 16; 1600 -> 4800 8.0 / 8.2, 9.5 / 8.5, 13.1 / 8.9;
    1600 -> 6400 8.3 / 8.8, 9.8 / 9.0, 13.2 / 9.3; 4096 -> 5120 13.7 / 15.2 at 4, 16.0 / 15.4 at 6.  And 5120 -> 2048 16.4 / 44.6 at 12."""
    if k_dim > 4096:
        return True
    if n_out > 4096:
        return n_rows * k_dim <= (16384 if k_dim == 4096 else 8192)
    if k_dim > 1024:
        if n_out * k_dim < (3_000_000 if k_dim <= 2048 else 2_700_000) and -(-n_out // 16) * -(-n_rows // 8) <= 256:
            return True
        return n_rows <= 4 if k_dim > 2048 else n_rows <= 8 or n_rows * k_dim <= 13000
    return n_rows <= 16 or n_out <= 2048 or k_dim < 768


def _rows_apart(ctx, plan, a: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], out: torch.Tensor, n_rows: int, epilogue: int,
                scatter) -> bool:
    """The product as kernels.linear_rows_plan says; False, with nothing launched, where the operands are not aligned for it."""
    shape, stretches = plan
    partials = None
    if stretches > 1:
        partials = ctx.workspace.get("linear_partials", stretches * n_rows * w.shape[0], 1, torch.float32)
    return kernels.linear_mfma(a, w, bias, out, n_rows, epilogue, scatter=scatter, shape=shape, partials=partials, k_parts=stretches)


def as_tensor(ctx, a: Union[torch.Tensor, LazyNorm]) -> torch.Tensor:
    return a.tensor(ctx) if isinstance(a, LazyNorm) else a


class TileBest:
    """Asks a product for the best column of every tile of 16 beside its float32 output: the largest
    value among the columns below `limit` and its column.  The product that can, fills values and
    columns ([rows, out / 16], from the workspace) and sets `filled`."""

    def __init__(self, limit: int) -> None:
        self.limit = int(limit)
        self.values: Optional[torch.Tensor] = None
        self.columns: Optional[torch.Tensor] = None
        self.filled = False


# A split product's parts are left pending for rows this wide, or this many: the LayerNorm kernel
# that then adds them up is one workgroup per row, and for one narrow row costs more than the
# kernel that adds the parts plus the folded LayerNorm it replaces (decode steps on one box, us:
# width 768: 296 against 284 at one row, 333 against 336 at 8, 365 against 369 at 16; width 1600:
# 1748 against 1768, 2049 against 2102, 2439 against 2554)
LEAVE_PARTS_MIN_WIDTH = 1024
LEAVE_PARTS_MIN_ROWS = 8
LEAVE_PARTS_MAX_ROWS = 256     # (the tiled kernel's split; the decode kernel's ends at its 64 rows)


# The 32-bit path leaves the sums over the product's blocks of k where that and the LayerNorm which adds them up take less than
# the product and a plain LayerNorm.
# us, product and LayerNorm / sums and LayerNorm: 768 -> 768 7.4 / 8.2 at 4 rows, 8.1 / 8.4 at 16, 8.4 / 8.6 at 64, 8.6 / 8.8 at 80, and from
# the row on from which the product's workgroups of 16 x 16 outputs are more than compute units 11.1 / 8.9 at 96, 14.5 / 10.3 at 176,
# 11.4 / 10.8 at 224, 11.6 / 12.8 at 256; 768 -> 512 7.3 / 7.8 at 4, 8.4 / 8.0 at 32, 8.6 / 8.8 at 128, 11.1 / 9.2 at 160.  1024 -> 1024 8.5 / 8.6
# at 8, 9.1 / 8.6 at 16, 14.9 / 14.8 at 224; 1280 -> 1280 9.4 / 8.7 at 1, 10.7 / 9.2 at 16, 17.3 / 15.8 at 160, 17.2 / 18.3 at 176, 22.0 / 19.0 at
# 224; 1600 -> 1600 9.8 / 9.3 at 1, 17.8 / 14.4 at 64, 26.9 / 25.5 at 224, 27.2 / 27.6 at 256; 2048 -> 512 9.6 / 7.8 at 1, 20.1 / 14.4 at 256;
# 2048 -> 2048 30.8 / 29.5 at 176, 30.6 / 31.4 at 192; 3072 -> 768 12.2 / 8.1 at 1, 18.0 / 12.8 at 64, 32.2 / 24.3 at 256; 6400 -> 1600 23.4 /
# 15.8 at 1, 49.7 / 27.0 at 64, 81.2 / 67.2 at 224.  That is with the matrix in the caches; read from memory, as in a decode step of a
# GPT-2-small shape (12 layers, 50,257 tokens), what sums gain a layer at 768 -> 768 is -1.2 us at 1 row, -0.7 at 8, 0.4 to 0.9 at 16
# (the step of 16 sampled requests 748 -> 738 us), 0 at 24 to 32, -0.4 at 48 to 64, 0.1 at 128; at 960 -> 960 -0.3 at 4, 1.0 at 16, 0.2 at 32,
# -0.3 at 64, 0.8 at 160.  So they are left at 13 to 16 rows too, where the product has least of the chip.
EXACT_PARTS_MAX_ROWS = 256
EXACT_PARTS_MAX_OUTPUTS = 380_000
EXACT_PARTS_SHORT_MAX_OUTPUTS = 172_000    # under inner sizes below 1,024


def exact_leaves_parts(n_rows: int, n_out: int, k_dim: int) -> bool:
    """Whether the 32-bit path leaves a product of this size as sums over its blocks of k for the LayerNorm behind it."""
    if k_dim < 768 or n_rows > EXACT_PARTS_MAX_ROWS:
        return False
    if k_dim < 1024:
        pays = 12 < n_rows <= 16 or -(-n_rows // 16) * -(-n_out // 16) > 256
        return pays and n_rows * n_out <= EXACT_PARTS_SHORT_MAX_OUTPUTS
    return n_rows >= (1 if k_dim >= 1280 else 16) and n_rows * n_out <= EXACT_PARTS_MAX_OUTPUTS


def plain_residual(ctx, h, x: torch.Tensor) -> None:
    """Makes the residual rows x plain for a part that reads or adds to them with ordinary kernels.
    If they are still a sum and h is the LayerNorm of them that the part is about to read, that
    LayerNorm is computed now: its kernel adds the sum up and stores it on the way."""
    if getattr(ctx, "pending", None) is None:
        return
    if isinstance(h, LazyNorm) and h.x is x and h._tensor is None:
        h.tensor(ctx)
    residual.settle(ctx, x, ctx.n_rows)


def linear_add(ctx, a: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], x: torch.Tensor, n_rows: int,
               may_leave_parts: bool = False) -> None:
    """x[:n_rows] += a[:n_rows] @ w.T (+ bias), x the float32 residual stream.

    may_leave_parts: the caller and whoever reads x next know of ctx.pending.  Then a product whose
    long inner size is split over workgroups anyway (few rows, few column tiles) leaves the
    workgroups' sums as the parts of a pending residual instead of running a second kernel that adds
    them into x; the LayerNorm that reads x next adds them up (LazyNorm.tensor).  The 32-bit path does so with the sums over
    the blocks of k that its products are made of, which has the bits of adding into x at once."""
    if (may_leave_parts and ctx.exact and getattr(ctx, "pending", None) is None and n_rows == ctx.n_rows
            and exact_leaves_parts(n_rows, *w.shape) and x.is_contiguous() and x.shape[1] == w.shape[0]
            and kernels.linear_exact_takes_parts(a, w, bias, x)):
        n_parts = kernels.linear_exact_blocks(w.shape[1])
        buf = ctx.workspace.get("residual_parts", n_parts * n_rows, w.shape[0], torch.float32)
        parts = buf[:n_parts * n_rows].view(n_parts, n_rows, w.shape[0])
        kernels.linear_exact_parts(a, w, parts, n_rows)
        ctx.pending = residual.PendingSums(x, parts, n_parts, exact=True, bias=bias)
        return
    leave = (may_leave_parts and getattr(ctx, "pending", None) is None and not ctx.exact
             and ctx.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and a.dtype == torch.bfloat16
             and 0 < n_rows <= LEAVE_PARTS_MAX_ROWS and n_rows == ctx.n_rows and x.is_contiguous()
             and x.shape[1] == w.shape[0] and w.shape[1] % 16 == 0)
    plan = kernels.linear_rows_plan(n_rows, *w.shape) if leave and n_rows <= 32 else None
    if plan is not None:
        # the sums of the kernel for few rows, where it cuts the inner size
        if 1 < plan[1] <= kernels.residual_parts_limit(w.shape[0]):
            buf = ctx.workspace.get("residual_parts", plan[1] * n_rows, w.shape[0], torch.float32)
            parts = buf[:plan[1] * n_rows].view(plan[1], n_rows, w.shape[0])
            if kernels.linear_mfma_parts(a, w, bias, parts, n_rows, plan):
                ctx.pending = residual.PendingSums(x, parts, plan[1])
                return
    elif leave and tiled_at_few_rows(n_rows, w, left=True):
        # the tiled kernel's split: its stretches' sums are the parts (2 to 8 of them)
        need = kernels.linear_mfma_partials(n_rows, w.shape[0], w.shape[1], kernels.EPI_RESIDUAL)
        n_parts = need // (n_rows * w.shape[0])
        if 1 < n_parts <= kernels.residual_parts_limit(w.shape[0]):
            buf = ctx.workspace.get("residual_parts", n_parts * n_rows, w.shape[0], torch.float32)
            parts = buf[:n_parts * n_rows].view(n_parts, n_rows, w.shape[0])
            if kernels.linear_mfma_parts(a, w, bias, parts, n_rows):
                ctx.pending = residual.PendingSums(x, parts, n_parts)
                return
    elif (leave and n_rows <= 64 and (w.shape[0] >= LEAVE_PARTS_MIN_WIDTH or n_rows >= LEAVE_PARTS_MIN_ROWS)
            and kernels.residual_parts_limit(w.shape[0]) >= 4
            and kernels.linear_skinny_partials(n_rows, w.shape[0], w.shape[1], False, kernels.EPI_RESIDUAL)):
        buf = ctx.workspace.get("residual_parts", 4 * n_rows, w.shape[0], torch.float32)
        parts = buf[:4 * n_rows].view(4, n_rows, w.shape[0])
        n_parts = kernels.linear_decode_parts(a, w, bias, parts, n_rows, w_packed=packed_weight(w, ctx))
        if n_parts:
            assert n_parts == 4
            ctx.pending = residual.PendingSums(x, parts, n_parts)
            return
    linear(ctx, a, w, bias, x, n_rows, kernels.EPI_RESIDUAL)


def linear_xielu(ctx, a: Union[torch.Tensor, LazyNorm], w: torch.Tensor, bias: Optional[torch.Tensor], out: torch.Tensor,
                 n_rows: int, coef: torch.Tensor) -> None:
    """out[:n_rows] = xielu(a[:n_rows] @ w.T (+ bias)) with the activation's two coefficients in `coef` (float32
    [2]).  Where the product goes to the tiled MFMA kernel (steps of many rows, and few rows under a large matrix)
    the activation is that kernel's epilogue; everywhere else (the decode kernel, the 32-bit path) it is a kernel of
    its own behind the product, in place."""
    if n_rows == 0:
        return
    fast = (w.dtype == torch.bfloat16 and not ctx.exact and ctx.dtype == torch.bfloat16 and w.shape[1] % 16 == 0
            and out.dtype == torch.bfloat16)
    wide_out = w.shape[0] >= WIDE_OUT and n_rows * w.shape[1] > WIDE_OUT_DECODE_WORK
    if fast and not (n_rows <= 64 and not wide_out and not tiled_at_few_rows(n_rows, w)):
        a = as_tensor(ctx, a)
        need = kernels.linear_mfma_partials(n_rows, w.shape[0], w.shape[1], kernels.EPI_XIELU)
        partials = ctx.workspace.get("linear_partials", need, 1, torch.float32) if need else None
        if kernels.linear_mfma_xielu(a, w, bias, out, n_rows, coef, partials=partials):
            return
    linear(ctx, a, w, bias, out, n_rows)
    kernels.xielu(out, out, coef, n_rows, w.shape[0], fast=not ctx.exact)


def linear(ctx, a: Union[torch.Tensor, LazyNorm], w: torch.Tensor, bias: Optional[torch.Tensor],
           out: torch.Tensor, n_rows: int, epilogue: int = kernels.EPI_NONE, scatter=None,
           tile_best: Optional[TileBest] = None) -> bool:
    """out[:n_rows] = a[:n_rows] @ w.T (+ bias) with the epilogue.

    On the bfloat16 path up to 32 rows under all but small matrices and very wide outputs go to the kernel that has nothing but them and a
    few columns a workgroup; else up to 64 rows (fewer for a very wide output) to the decode step's MFMA kernels (reading the residual
    stream through the folded LayerNorm when `a` is a LazyNorm of a fusable norm and the rows are
    few; splitting a long inner size over workgroups when the rows are many) and more rows to the
    tiled MFMA kernel (which also splits a long inner size when its tiles are few); the 32-bit path, and every shape those refuse, go to the general product
    (on the matrix cores in 32 bits where everything is float32; at few rows with the LayerNorm of a LazyNorm inside).  `scatter` = (k_pool, v_pool,
    slot_mapping, q_width, kv_width) asks for the new keys and values to be stored into their
    pages by the same kernel; the return value says whether that was done."""
    if n_rows == 0:
        return scatter is not None
    if isinstance(a, LazyNorm) and getattr(ctx, "pending", None) is not None:
        a = a.tensor(ctx)      # the kernels below read plain residual rows
    # (the MFMA kernels take inner sizes in steps of 16; any other goes to the general kernel)
    fast = w.dtype == torch.bfloat16 and not ctx.exact and ctx.dtype == torch.bfloat16 and w.shape[1] % 16 == 0
    wide_out = w.shape[0] >= WIDE_OUT and n_rows * w.shape[1] > WIDE_OUT_DECODE_WORK
    if (tile_best is not None and fast and n_rows <= 16 and not wide_out and epilogue == kernels.EPI_NONE
            and scatter is None and w.shape[0] % 16 == 0 and w.shape[1] % 32 == 0
            and not kernels.linear_skinny_partials(n_rows, w.shape[0], w.shape[1], False, epilogue)):
        rows = out.shape[0]
        tile_best.values = ctx.workspace.get("tile_best_values", rows, w.shape[0] // 16, torch.float32)
        tile_best.columns = ctx.workspace.get("tile_best_columns", rows, w.shape[0] // 16, torch.int32)
        if kernels.linear_head_best(as_tensor(ctx, a), w, bias, out, n_rows, tile_best.values, tile_best.columns,
                                    tile_best.limit, w_packed=packed_weight(w, ctx)):
            tile_best.filled = True
            return False
    plan = kernels.linear_rows_plan(n_rows, *w.shape, scatter is not None) if fast and n_rows <= 32 and not wide_out else None
    if fast and n_rows <= 64 and not wide_out and not tiled_at_few_rows(n_rows, w):
        epi = kernels.SK_EPI_QKV if scatter is not None else epilogue
        if (isinstance(a, LazyNorm) and getattr(a.norm, "fusable_layer_norm", False) and a._tensor is None
                and (plan is None or folds_before_rows_apart(n_rows, *w.shape))
                and (w.shape[0] <= FOLD_MAX_OUT
                     or (n_rows <= FOLD_ANY_OUT_MAX_ROWS and w.shape[0] <= FOLD_ANY_OUT_MAX_OUT))
                and (n_rows <= FOLD_MAX_ROWS or kernels.linear_skinny_row_groups(n_rows, w.shape[0], w.shape[1]))):
            folded = folded_layer_norm(a.norm, w, bias, ctx)
            if folded is not None:
                wf, colsum, bias_f = folded
                if kernels.linear_skinny(None, wf, bias_f, out, n_rows, epi, ln_x=a.x, ln_colsum=colsum,
                                         ln_eps=a.norm.eps, ln_rows=a.rows, scatter=scatter,
                                         w_packed=packed_weight(wf, ctx)):
                    return scatter is not None
        if plan is not None and _rows_apart(ctx, plan, as_tensor(ctx, a), w, bias, out, n_rows, epilogue, scatter):
            return scatter is not None
        partials = None
        need = kernels.linear_skinny_partials(n_rows, w.shape[0], w.shape[1], False, epi)
        if need:
            partials = ctx.workspace.get("linear_partials", need, 1, torch.float32)
        if kernels.linear_skinny(as_tensor(ctx, a), w, bias, out, n_rows, epi, scatter=scatter, partials=partials,
                                 w_packed=packed_weight(w, ctx)):
            return scatter is not None
    if (isinstance(a, LazyNorm) and ctx.exact and a._tensor is None and getattr(a.norm, "fusable_layer_norm", False)
            and a.x.is_contiguous()
            and kernels.linear_exact_normed(a.x, a.norm.weight, a.norm.bias, a.norm.eps, w, bias, out, n_rows, epilogue, a.rows,
                                            scatter)):
        return scatter is not None
    a = as_tensor(ctx, a)
    if (fast and wide_out and bias is None and scatter is None and epilogue == kernels.EPI_NONE and wide_rows_once(n_rows, *w.shape)
            and kernels.linear_rows_once(a, w, out, n_rows)):
        return False
    if plan is not None and _rows_apart(ctx, plan, a, w, bias, out, n_rows, epilogue, scatter):
        return scatter is not None
    if fast and scatter is not None and kernels.linear_mfma(a, w, bias, out, n_rows, epilogue, scatter=scatter):
        return True
    if fast:
        need = kernels.linear_mfma_partials(n_rows, w.shape[0], w.shape[1], epilogue)
        partials = ctx.workspace.get("linear_partials", need, 1, torch.float32) if need else None
        if kernels.linear_mfma(a, w, bias, out, n_rows, epilogue, partials=partials):
            return False
    if scatter is not None and epilogue == kernels.EPI_NONE and kernels.linear_exact_qkv(a, w, bias, out, n_rows, scatter):
        return True
    kernels.linear_generic(a, w, bias, out, n_rows, epilogue)
    return False
