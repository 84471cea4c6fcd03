"""Chooses the matrix-product kernel for a linear layer by dtype and shape."""

from __future__ import annotations

import torch

from . import ops

SKINNY_MAX_ROWS = 64   # what the skinny MFMA kernel takes
SKINNY_ROWS = 64       # up to here the few-rows kernels run; beyond, the many-rows kernel (ops.linear_big)


LONG_K = 8192            # a K that the split-K kernel cuts into eight pieces of sixteen chunks
FEW_COLUMNS_PER_UNIT = 32     # up to this many columns per compute unit the few-rows kernel has two workgroups a unit at most
MANY_COLUMNS_PER_UNIT = 64    # from this many on its workgroups come in several rounds, each reading all of x again


def _mid_is_faster(m: int, n: int, k: int) -> bool:
    """From 17 rows on, the kernel that shares x inside a workgroup and splits K over workgroups wins where K is
    long and the columns are few for the device (7B down projection on 256 units: 26 + 5 us against 38 at 32 rows,
    34 + 5 against 53 at 64) and where there are very many columns (gate_up: steps of 20 to 32 requests 1.7 %
    shorter, 58 + 8 us against 79 at 64 rows).  Measured inside decode steps at 7B layer sizes; the bounds on the
    columns go with the device's compute units."""
    if m <= 16:
        return False
    units = ops.compute_units()
    return (k >= LONG_K and n <= FEW_COLUMNS_PER_UNIT * units) or n >= MANY_COLUMNS_PER_UNIT * units


FEW_ROWS = ops.FUSED_ROWS
SMALL_PRODUCT = 4096          # 16-column strips of 64 rows times K, a compute unit: up to here blocks of 64 rows win
NEXT_PRODUCT = 8192           # up to here with few blocks, or all at once


def few_rows(m: int, n: int, k: int) -> bool:
    """Whether the few-rows products that are fused with the stream and the norm take this many rows: up to 64 always, more in
    blocks of 64 where the product is small for the device.  The many-rows kernel has 256-column tiles there that leave most
    of the device idle, a second launch that adds the sums of its K splits and one for the rows' scales.  Measured
    at 128 rows (many rows / blocks, us, with those launches): 0.5B q/k/v 21 / 8.1, o 17 / 5.1, gate_up 23 / 16, down
    22 / 10.9; 7B q/k/v 34 / 27, o 27 / 21, but gate_up 68 / 138; at 768 rows 0.5B q/k/v 25 / 17, o 19 / 16, down
    28 / 44.  The work of a compute unit, in strips of 16 columns by 64 rows by K, tells them apart: 0.5B down
    loses from 5 blocks (5,320), 7B o from 3 (9,408), a 14B layer's q/k/v at once (17,920)."""
    if m <= FEW_ROWS:
        return True
    blocks, strips, units = (m + FEW_ROWS - 1) // FEW_ROWS, (n + 15) // 16, ops.compute_units()
    if m > ops.FUSED_MAX_ROWS:
        return False
    share = blocks * strips * k / units
    return share <= SMALL_PRODUCT or (share <= NEXT_PRODUCT and (blocks <= 3 or blocks * strips <= units))


EVEN_COLUMNS_PER_UNIT = 192   # the widest workgroup of the kernel that deals columns out evenly
EVEN_LONG_K_ROWS = 49         # from here the product with a long K into the stream takes the kernel with even shares of columns
EVEN_WEIGHTS_PER_UNIT = 131072    # and, up to 64 rows, from this many weights a compute unit


def even_gated(m: int, n: int, k: int) -> bool:
    """Whether a scaled, gated product of 17 to 192 rows takes the kernel that deals its columns out evenly over the compute units:
    where they are more than 64 a unit and fit into one round of its workgroups, of up to 192 columns (37,888 columns at
    17 / 64 / 128 rows 45 / 51 / 63 us against 55 / 63 / 68 of the kernels below and beyond 64 rows; 17,920 15 / 21 / 25 against
    18 / 23 / 34).  16,384 columns are one whole round of the kernel that splits K (64 rows: 31 against 27), fewer leave units
    without a workgroup, and up to 16 rows the few-rows kernel is ahead (37,888 columns, 8 rows: 44.6 against 48).  In two
    rounds it is ahead only up to 64 rows with inputs a multiple of 4 KB (57,344 x 8,192 at 64 rows 156 against 195; at 128 rows 182
    against 160; 55,296 x 5,120 at 64 rows 111 against 106).  Beyond 128 rows the many-rows kernel's 192-row tiles of 128 columns
    are ahead as long as they are one round (27,648 columns at 160 rows 79 against 82; 37,888 86 against 73)."""
    per_unit = n / ops.compute_units()
    if m <= 16 or m > ops.EVEN_MAX_ROWS or per_unit <= (MANY_COLUMNS_PER_UNIT if m <= 128 else 2 * MANY_COLUMNS_PER_UNIT):
        return False
    return per_unit <= EVEN_COLUMNS_PER_UNIT or (m <= FEW_ROWS and k % 2048 == 0)


def even_residual(m: int, n: int, k: int) -> bool:
    """The same for the product into the stream, where K is long and the columns few: 3,584 x 18,944 at 17 / 48 / 64 / 128 rows
    27.5 / 30.9 / 32.4 / 40 us against 26.8 / 32.0 / 35.7 / 51.  Up to 64 rows a smaller weight stays with the few-rows kernels
    (2,048 x 11,008 at 64 rows 19.4 against 17.9, 1,536 x 8,960 17.5 against 13.9); beyond, their blocks of 64 and the many-rows
    kernel take longer (20 and 18 against 29 and 26 at 65 rows)."""
    units = ops.compute_units()
    return (EVEN_LONG_K_ROWS <= m <= 128 and k >= LONG_K and n <= FEW_COLUMNS_PER_UNIT * units
            and (m > FEW_ROWS or n * k >= EVEN_WEIGHTS_PER_UNIT * units))


def linear_swiglu(x: torch.Tensor, weight: torch.Tensor, activation: str = "silu") -> torch.Tensor:
    """act(x @ gate.T) * (x @ up.T) for bfloat16 rows, act "silu" or "gelu_tanh"; weight: [2 I, K], gate and up rows
    interleaved in blocks of 16."""
    m, k = x.shape
    if m > SKINNY_ROWS:
        return ops.linear_big(x, weight, swiglu=activation)
    if _mid_is_faster(m, weight.shape[0], k):
        return ops.linear_mid(x, weight, swiglu=activation)
    return ops.linear_skinny_swiglu(x, weight, activation)


def linear_residual(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, h: torch.Tensor,
                    next_norm_weight: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor | None]:
    """h += x @ weight.T (+ bias) in place, by the kernel that :func:`linear` would take for the sizes; see
    :func:`ops.linear_residual`.  Rows beyond :func:`few_rows` take the many-rows kernel, which shares a tile's K among workgroups
    where its tiles are few (o and down of 65 to some hundred rows; passes of the few-rows kernel over 64 rows each
    measured the same inside decode steps of 128 requests, 10.70 against 10.72 ms)."""
    m, n = x.shape[0], weight.shape[0]
    if even_residual(m, n, x.shape[1]) and ops.even_supported(x, weight, h):
        return ops.linear_even_residual(x, weight, bias, h, next_norm_weight)
    if not few_rows(m, n, x.shape[1]):
        return ops.linear_big_residual(x, weight, bias, h, next_norm_weight)
    mid = m <= FEW_ROWS and _mid_is_faster(m, n, x.shape[1])
    return ops.linear_residual(x, weight, bias, h, next_norm_weight, mid=mid, row_blocks=True)


def linear_scaled(x: torch.Tensor, eps: float, stats: torch.Tensor, weight: torch.Tensor,
                  bias: torch.Tensor | None = None, swiglu: "bool | str" = False) -> torch.Tensor:
    """The product of rows that are still to be normed, by the kernel that :func:`linear` would take for the
    sizes; see :func:`ops.linear_scaled`."""
    if swiglu and bias is None and even_gated(x.shape[0], weight.shape[0], x.shape[1]) and ops.even_supported(x, weight, stats):
        return ops.linear_even_gated(x, eps, stats, weight, swiglu)
    if not few_rows(x.shape[0], weight.shape[0], x.shape[1]):
        return ops.linear_big(x, weight, bias, swiglu=swiglu, eps=eps, stats=stats)
    mid = x.shape[0] <= FEW_ROWS and _mid_is_faster(x.shape[0], weight.shape[0], x.shape[1])
    return ops.linear_scaled(x, eps, stats, weight, bias, swiglu, mid=mid, row_blocks=True)


def linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None = None,
           out_dtype: torch.dtype | None = None) -> torch.Tensor:
    """x @ weight.T (+ bias).

    float32 takes the float32 matrix-core kernel (the true 32-bit path; the plain FMA kernel where K is no multiple of 4: the
    weight alone decides, so that every number of rows runs one of the two).  bfloat16 with few rows takes the
    hand-written few-rows MFMA kernels, with more rows the many-rows MFMA kernel (256-row tiles), whose float32
    form writes the logits of many rows without rounding them to bfloat16 (rows of an input it does not take go
    through the few-rows kernel 64 at a time).  Operands the MFMA kernels do not take (K no multiple of 8, unaligned) run the plain
    kernel.
    """
    out_dtype = out_dtype or x.dtype
    if x.dtype == torch.float32:
        if out_dtype == torch.float32 and ops.linear_f32_supported(weight):
            return ops.linear_f32(x, weight, bias)
        return ops.linear_plain(x, weight, bias, out_dtype)
    m, k = x.shape
    if k % 8 != 0 or x.data_ptr() % 16 or weight.data_ptr() % 16:
        return ops.linear_plain(x, weight, bias, out_dtype)
    if m <= SKINNY_ROWS:
        if _mid_is_faster(m, weight.shape[0], k):
            return ops.linear_mid(x, weight, bias, out_dtype)
        return ops.linear_skinny(x, weight, bias, out_dtype)
    if out_dtype == x.dtype and ops.big_supported(x, weight):
        return ops.linear_big(x, weight, bias)
    if out_dtype == torch.float32 and ops.big_supported(x, weight):
        # logits of more than 64 rows: one pass over the output matrix instead of one per 64 rows (7B head at 256 rows:
        # four passes of 290 us)
        return ops.linear_big_f32(x, weight, bias)
    if out_dtype == torch.float32:
        return torch.cat([ops.linear_skinny(x[at:at + SKINNY_MAX_ROWS], weight, bias, out_dtype)
                          for at in range(0, m, SKINNY_MAX_ROWS)])
    return ops.linear_plain(x, weight, bias, out_dtype)
