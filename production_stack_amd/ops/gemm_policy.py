"""Per-shape GEMM dispatch: hipBLASLt (torch F.linear) vs the in-house
skinny split-K MFMA kernel.

The library's decode-shaped tiles leave the read of the weights at a third to
a half of memory's rate for several projections, csrc/skinny_gemm.hip does for
others: the engine autotunes each (decode bucket M, projection
shape) pair once at startup on the actual device and the winner is what the
hipGraph capture records. That times bare products. Where a launch before or
behind one can be joined with it, the rules below, which were measured with those
launches, decide first.
"""

from __future__ import annotations

import logging
import math
import time
from typing import Dict

import torch
import torch.nn.functional as F

logger = logging.getLogger("ops.gemm_policy")

# (M, N, K) -> winning impl: 0 = hipBLASLt, 1 = skinny split-K, 2 = 8-phase;
# (M, N, K, behind) -> that of a product joined with other launches
_POLICY: Dict[tuple, int] = {}


MAX_ROWS = 256  # of the skinny kernels


def _eligible(M: int, N: int, K: int) -> bool:
    return M <= MAX_ROWS and N % 64 == 0 and K % 64 == 0


def _eligible_8p(M: int, N: int, K: int) -> bool:
    return N % 256 == 0 and K % 128 == 0


def _time_fn(fn, iters: int = 20) -> float:
    for _ in range(3):
        fn()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(iters):
        fn()
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) / iters


def tune(weights, buckets, device) -> None:
    """weights: iterable of weight tensors [N, K]; buckets: decode batch
    sizes to tune for."""
    from production_stack_amd import ops

    shapes = sorted({(int(w.shape[0]), int(w.shape[1])) for w in weights})
    w_by_shape = {}
    for w in weights:
        w_by_shape.setdefault((int(w.shape[0]), int(w.shape[1])), w)
    for M in buckets:
        for (N, K) in shapes:
            w = w_by_shape[(N, K)]
            x = torch.randn(M, K, dtype=torch.bfloat16, device=device)
            cands = [(0, _time_fn(lambda: F.linear(x, w)))]
            if _eligible(M, N, K):
                cands.append((1, _time_fn(lambda: ops.skinny_gemm(x, w))))
            if _eligible_8p(M, N, K):
                cands.append((2, _time_fn(lambda: ops.gemm8p(x, w))))
            impl, t = min(cands, key=lambda c: c[1])
            _POLICY[(M, N, K)] = impl
            for behind, rules in _UNTUNED.items():
                if behind:
                    _POLICY[(M, N, K, behind)] = (
                        1 if any(rule(M, N, K) for rule in rules) else impl)
            if impl:
                logger.info(
                    "gemm M=%d N=%d K=%d: impl %s wins at %.1fus",
                    M, N, K, ("blas", "skinny", "8p")[impl], t * 1e6,
                )
    cells = [v for key, v in _POLICY.items() if len(key) == 3]
    logger.info(
        "gemm autotune done: %d/%d cells use an in-house kernel",
        sum(1 for v in cells if v), len(cells),
    )


def _fits(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Operands that the in-house kernel takes as they are."""
    from production_stack_amd import ops

    return (x.dim() == 2 and x.shape[0] > 0
            and _eligible(x.shape[0], *w.shape) and x.stride(1) == 1
            and x.shape[1] == w.shape[1] and w.dtype == torch.bfloat16
            and w.is_contiguous() and x.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and ops.HAVE_EXT
            and not (torch.is_grad_enabled()
                     and (x.requires_grad or w.requires_grad)))


# entries of x that the kernel with x in LDS takes, with the norm and without
_LDS_X, _LDS_NORM_X = 65536, 16384


def _few_rows(rows: int, N: int, K: int) -> bool:
    """Up to 16 rows, x of up to 65536 entries. Rows of W of up to 4096 entries
    (us, in-house / library: 1 x 2048 x 2048 4.5 / 11.0, 1 x 28672 x 4096 41 / 63,
    16 x 28672 x 4096 45 / 64, 16 x 4096 x 4096 10.6 / 15.4, 16 x 6144 x 4096 14.4 /
    15.5, 16 x 6144 x 2560 10.1 / 10.5, 16 x 128256 x 4096 189 / 191; the narrowest;
    past the line 1 x 50304 x 768 18.1 / 15.8, 16 x 50304 x 768 19.1 / 16.0), and longer ones of up to 2048 rows of W (8 x 2048 x 8192 10.5 / 12.6, 8 x 512 x
    8192 10.0 / 11.4; 16 x 2048 x 8192 16.8 / 12.9) or, up to 4 rows, of as many as
    give all CUs nearly as much to do (4 x 4096 x 14336 25.8 / 27.0, 4 x 28672 x 8192
    82 / 122, 1 x 4096 x 8192 15.2 / 16.2; past the line 4 x 6144 x 8192 24 / 22, 4 x
    5120 x 8192 23 / 20)."""
    if rows > 16 or rows * K > _LDS_X:
        return False
    if K <= 4096:
        return K > 1024 or N < 32768
    if N <= 2048:
        return rows <= 8 and K % 128 == 0
    turns = N / 4096
    return rows <= 4 and turns >= 0.8 * math.ceil(turns)


def _long_rows(rows: int, N: int, K: int) -> bool:
    """48 to 192 rows (24 where rows of W have 14336 entries) of a W of few long
    rows, whose tiles fill the chip only in ranges of K. us, in-house / library:
    4096 x 14336 with 24 rows 28.5 / 31.3, 64 31.3 / 38.3, 128 38.4 / 73.8, 192
    46.2 / 100; 2560 x 10240 with 48 20.9 / 21.5, 128 26.6 / 54.5; 8192 x 28672 with
    64 96 / 147; 2048 x 16384 with 40 22.0 / 26.7. Past the lines 2048 x 10240 with
    40 18.3 / 17.5, 4096 x 12288 with 24 25.8 / 23.9, 8192 x 13824 with 32 47.5 / 45.0,
    6144 x 12288 with 20 36.3 / 34.5, 4096 x 11008 with 208 49.8 / 45.5, 1024 x 10240
    with 80 19.9 / 18.2, 10240 x 8192 with 64 42.6 / 41.4, 4096 x 8192 with 160 31.6 /
    32.3 (128 rows 29 / 32). No wide tiles, so slower, where N is no multiple of
    128: 6464 x 13568 with 88 70.1 / 56.6, 5184 x 12672 with 184 73.0 / 60.2. The
    slowest found within: 6784 x 15360 with 28 45.4 / 43.0."""
    return ((24 if K >= 14336 else 48) <= rows <= 192
            and 2048 <= N <= 8192 and N % 128 == 0 and K >= 10240)


def _rows_before_norm(rows: int, N: int, K: int) -> bool:
    """17 to 192 rows whose partial sums the norm behind them adds. us with that
    norm, in-house / library: 17 x 2048 x 2048 10.1 / 13.8, 64 x 2048 x 8192 18.4 /
    25.2, 64 x 4096 x 4096 17.0 / 18.4, 192 x 4096 x 4096 24.9 / 36.3, 64 x 4096 x
    14336 32.7 / 42.5, 96 x 3584 x 4096 20.1 / 25.3, 128 x 6144 x 4096 27.2 / 29.6,
    192 x 8192 x 14336 78 / 117. Past the lines 64 x 6144 x 4096 22.7 / 22.0, 17 x
    2048 x 8192 16.8 / 16.5, 96 x 2560 x 4096 19.4 / 16.3, 160 x 3072 x 4096 22.5 /
    20.2, 128 x 4096 x 2048 18.8 / 18.7, 256 x 4096 x 8192 45.6 / 40.1. The slowest
    found within: 48 x 2560 x 2560 13.7 / 12.7."""
    if not 17 <= rows <= 192 or not 1024 <= N <= 8192 or K < 1024:
        return False
    if K >= 10240:
        return True
    if rows > 64:
        return 3584 <= N <= 6144 and K >= 4096
    return N <= 4096 and (K <= 5120 or (rows >= 48 and N >= 1536))


def _rows_before_rope(rows: int, N: int, K: int) -> bool:
    """As above with the rotary embedding and the cache's rows behind: 128 x 6144 x
    4096 27.0 / 28.6, 192 32.0 / 37.0, 128 x 7168 x 5120 35.3 / 36.7, 128 x 4608 x 3584
    24.6 / 26.1; past the lines 96 x 4608 x 3584 23.6 / 23.4, 192 x 6144 x 2048 26.2 /
    25.8, 160 x 3072 x 2048 21.6 / 15.9."""
    return 128 <= rows <= 192 and 4608 <= N <= 10240 and K >= 3584


def _rows_before_gate(rows: int, N: int, K: int) -> bool:
    """As above with the activation behind, in tiles that have all of K and fill
    the CUs once, rows of W a power of two apart or nearly (where the library is
    slow): 17 x 28672 x 4096 49.5 / 56.4, 64 51.7 / 55.4, 64 x 28672 x 2048 30.7 / 33.1,
    64 x 32768 x 8192 105 / 123; past the lines 96 x 28672 x 4096 59.5 / 56.3, 64 x
    24576 x 4096 50.8 / 49.0, 17 x 28672 x 2560 36.6 / 31.7, 64 x 57344 x 4096 106 /
    102."""
    return 17 <= rows <= 64 and 28160 <= N <= 32768 and K % 2048 == 0


_UNTUNED = {"": (_few_rows, _long_rows),
            "around": (_few_rows,),
            "norm": (_rows_before_norm,),
            "rope": (_rows_before_rope,),
            "gate": (_few_rows, _long_rows, _rows_before_gate)}


def _choose(x: torch.Tensor, w: torch.Tensor, behind: str = "") -> int:
    """0: the library, 1: skinny, 2: 8-phase. behind: what the product's last step
    shares a launch with ("around": its first one too). A choice that was made for
    the bare product alone holds for that as well."""
    if not x.is_cuda or x.dtype != torch.bfloat16:
        return 0
    shape = (x.shape[0], w.shape[0], w.shape[1])
    impl = _POLICY.get(shape + (behind,) if behind else shape)
    if impl is None:
        impl = _POLICY.get(shape)
    if impl is None:  # untuned
        impl = int(any(rule(*shape) for rule in _UNTUNED[behind])
                   and _fits(x, w))
    return impl


def parts(x: torch.Tensor, w: torch.Tensor, behind: str):
    """linear(x, w) as partial sums in fp32 [splits, rows, columns] for "norm"
    (ops.add_rms_norm_parts) or "rope" (ops.rope_cache_parts) to add, or None
    where linear is to be called."""
    from production_stack_amd import ops

    if 16 < x.shape[0] <= MAX_ROWS and _choose(x, w, behind) == 1 and _fits(x, w):
        return ops.skinny_parts(x, w)
    return None


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear with autotuned dispatch (no bias; Llama has none). The
    in-house kernels are bfloat16 only; other types take the library."""
    impl = _choose(x, w)
    if impl:
        from production_stack_amd import ops

        return (ops.skinny_gemm if impl == 1 else ops.gemm8p)(x, w)
    return F.linear(x, w)


def fused(x: torch.Tensor, w: torch.Tensor) -> int:
    """What the launch of x @ w.T may have around it: 0 nothing, 1 the rotary
    embedding and the cache's rows behind it, 2 the residual's sum and the norm
    before it too. That is as many rows as LDS has room for (a launch of its own
    costs a decode step 3.5 us and up; the norm in every workgroup of 8 x 4096
    entries as much)."""
    if x.shape[0] > 16:
        return 0
    entries = x.shape[0] * x.shape[-1]
    if (entries > _LDS_X or _choose(x, w, "around") != 1
            or not _fits(x, w) or (w.shape[0] + 32) * w.shape[1] >= 1 << 31):
        return 0
    return 2 if entries <= _LDS_NORM_X and x.is_contiguous() else 1


def silu_mul(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """silu_and_mul(linear(x, w)). Up to 16 rows (8 of a W of more than 32768)
    that take the skinny kernel, and more where its tiles have all of K, have the
    activation in its last step (a launch of its own costs a decode step 4.5 us
    a layer and more)."""
    from production_stack_amd import ops

    rows = 8 if w.shape[0] > 32768 else 16
    if _choose(x, w, "gate") == 1 and _fits(x, w):
        if x.shape[0] <= rows:
            return ops.skinny_gated(x, w)
        if 16 < x.shape[0] <= 192:
            act = ops.skinny_gated_tiles(x, w)
            if act is not None:
                return act
    return ops.silu_and_mul(linear(x, w))


def norm_silu_mul(x: torch.Tensor, residual: torch.Tensor,
                  norm_w: torch.Tensor, eps: float, w: torch.Tensor):
    """(silu_mul(y, w), x + residual), y the RMSNorm of x + residual; x may be
    partial sums; x and residual may be overwritten."""
    from production_stack_amd import ops

    if x.dim() == 2 and fused(x, w) == 2 and residual.is_contiguous():
        return ops.skinny_norm_gated(x, residual, norm_w, eps, w)
    add_norm = (ops.fused_add_rms_norm if x.dim() == 2
                else ops.add_rms_norm_parts)
    x, residual = add_norm(x, residual, norm_w, eps)
    return silu_mul(x, w), residual


def reset() -> None:
    _POLICY.clear()
