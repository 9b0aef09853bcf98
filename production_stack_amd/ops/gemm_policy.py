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


_PASSES = 512 << 20  # bytes read between timed calls: twice the last cache


def _time_fn(fn, others=None, iters: int = 15) -> float:
    """Seconds of a call. others: a tensor that is read before each, so that
    weights come from memory as in a decode step, where the other layers' have
    passed through the caches. (A matrix that stays there made the skinny kernel
    win where it loses: steps of 16, 48, 96 and 144 rows of a 1b-sized stack 627,
    853, 1076 and 1346 us, 598, 823, 1054 and 1254 so.)"""
    for _ in range(3):
        fn()
    spans = []
    for _ in range(iters):
        if others is not None:
            others.max()  # fn is queued before this is done
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        fn()
        b.record()
        spans.append((a, b))
    torch.cuda.synchronize()
    return sorted(a.elapsed_time(b) for a, b in spans)[iters // 2] * 1e-3


def tune(weights, buckets, device) -> None:
    """weights: iterable of weight tensors [N, K]; buckets: decode batch
    sizes to tune for."""
    from production_stack_amd import ops

    shapes = sorted({(int(w.shape[0]), int(w.shape[1])) for w in weights})
    w_by_shape = {}
    for w in weights:
        w_by_shape.setdefault((int(w.shape[0]), int(w.shape[1])), w)
    try:
        others = torch.zeros(_PASSES // 4, dtype=torch.int32, device=device)
    except torch.cuda.OutOfMemoryError:
        others = None
    for M in buckets:
        for (N, K) in shapes:
            w = w_by_shape[(N, K)]
            x = torch.randn(M, K, dtype=torch.bfloat16, device=device)
            cands = [(0, _time_fn(lambda: F.linear(x, w), others))]
            if _eligible(M, N, K):
                cands.append((1, _time_fn(lambda: ops.skinny_gemm(x, w),
                                          others)))
            if _eligible_8p(M, N, K):
                cands.append((2, _time_fn(lambda: ops.gemm8p(x, w), others)))
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
    del others
    torch.cuda.empty_cache()
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


# entries of x that the kernel with x in LDS takes, without the norm and with it
# (what _C.skinny_limits() says)
_LDS_X, _LDS_NORM_X = 65536, 16384


def _few_rows(rows: int, N: int, K: int) -> bool:
    """Up to 16 rows, x of up to 65536 entries. Rows of W of up to 4096 entries
    (us, in-house / library: 1 x 2048 x 2048 4.5 / 11.0, 1 x 28672 x 4096 41 / 63,
    16 x 28672 x 4096 45 / 64, 16 x 4096 x 4096 10.6 / 15.4, 16 x 6144 x 2560 10.1 /
    10.5, 16 x 128256 x 4096 189 / 191; the narrowest), without short rows of a wide
    W (1 x 50304 x 768 18.1 / 15.8, 16 x 28672 x 256 9.6 / 8.3, 16 x 18432 x 192 7.0 /
    6.0), from 4 rows on also
    of other lengths than whole 1024 (16 x 128256 x 1536 82.7 / 74.3, 16 x 50304 x
    3584 69.6 / 65.2). Longer ones of up to 2048 rows of W (8 x 2048 x 8192 10.5 /
    12.6; 16 x 2048 x 8192 16.8 / 12.9, 8 x 256 x 8192 9.7 / 8.4) or, up to 4 rows, of
    as many as give all CUs nearly as much to do (4 x 4096 x 14336 25.8 / 27.0, 4 x
    28672 x 8192 82 / 122, 1 x 4096 x 8192 15.2 / 16.2; past the line 4 x 6144 x 8192
    24 / 22, 4 x 5120 x 8192 23 / 20)."""
    if rows > 16 or rows * K > _LDS_X:
        return False
    if K <= 4096:
        if N >= 32768:
            return K > 1024 and (rows <= 3 or K % 1024 == 0)
        return K >= 512 or N < (24576 if K >= 256 else 14336)
    if N <= 2048:
        return rows <= (8 if N >= 1024 else 5) and K % 128 == 0
    turns = N / 4096
    return rows <= 4 and turns >= 0.8 * math.ceil(turns)


def _few_rows_alone(rows: int, N: int, K: int) -> bool:
    """As above where nothing else shares the launch: at 13 to 16 rows, tiles that
    are more than the CUs and not many times as many (16 x 5120 x 4096 14.3 / 13.9, x
    3584 13.1 / 12.6, 16 x 8192 x 3584 14.4 / 14.0) are the library's."""
    return (_few_rows(rows, N, K)
            and not (rows > 12 and 4096 < N <= 8192 and K > 3072))


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
    norm, in-house / library; the library's time jumps up at whole 32 rows, and
    between its tuned sizes in N and K it is some other kernel's.
    Long rows: 64 x 4096 x 14336 33.3 / 43.7, 17 x 8192 x 10240 41.7 / 42.1, but 20 x
    8192 x 13824 51.3 / 47.0, 17 x 4096 x 12288 28.1 / 26.8, 104 x 1024 x 10240 21.6 /
    19.2.
    More than 64 rows: 96 x 4096 x 4096 21.4 / 25.3, 192 24.8 / 36.3, but 80 21.0 /
    19.9, 112 22.0 / 20.0; 144 24.0 / 25.5; 80 x 5120 x 4096 25.2 / 21.4, 112 26.1 /
    27.7, 149 x 5376 x 4096 28.4 / 27.1; 80 x 6144 x 4096 25.9 / 27.5, 144 30.8 /
    43.8, 176 1.02 times.
    Of few rows of W, long ones: 65 x 3072 x 8192 24.0 / 40.7, 112 26.6 / 30.9, 128 27.6
    / 46.2, 192 32.7 / 62.5 (decode steps of a 3b-sized stack of five layers 67 869 ->
    795, 128 1020 -> 942, 192 1270 -> 1135), 161 30.7 / 35.8, 176 31.6 / 37.5, 191 32.6 /
    37.8 (N 2944 to 3520, K 6144 to 10112: 161 to 191 rows 0.68 to 0.95 times), but 160
    31.0 / 31.8 and 129 x 3072 x 6144 26.7 / 26.2 (steps of 161, 176 and 191 rows 920 ->
    905, 1016 -> 1006, 988 -> 977); 67 x 2048 x 8192 20.2
    / 23.5 (65 598 -> 585). A step gains some 2 us a product less than these
    differences: 100 x 2048 x 8192 22.0 / 23.8, but steps 763 -> 769, 128 23.0 / 24.1
    and 796 -> 820; 160 x 3072 x 8192 993 -> 1005.
    Fewer: few rows of W (17 x 2048 x 2048 10.1 / 13.7, 63 x 2048 x 4096 14.2 / 15.0, 48
    x 2560 x 2048 13.5 / 14.8; 25 x 2048 x 1024 9.0 / 8.4, 60 x 1024 x 1280 up to 1.2
    times, 48 x 2560 x 2560 14.5 / 12.7), of more 64 x 4096 x 4096 17.6 / 18.6 and 32 x
    4096 x 4096 16.0 / 16.3, but 63 x 4096 x 4096 17.7 / 17.2, 32 x 4096 x 3072 14.7 /
    14.1, 64 x 3584 x 3328 18.2 / 16.7. Of 1950 drawn sizes within the slowest, 63 x
    1536 x 3072, takes 13.5 / 12.8."""
    if not 17 <= rows <= 192 or not 1024 <= N <= 8192 or K < 1024:
        return False
    whole = rows % 32 == 0
    if K >= 10240:
        return ((N >= 1536 or K >= 14336) and
                (rows >= 32 or (K % 2048 == 0 and
                                (K >= 14336 or not 3072 < N < 4608))))
    if rows > 64:
        if K >= 6144 and 2944 <= N < 3584:
            return rows <= 128 or rows > 160
        if K >= 7168 and 2048 <= N <= 2112:
            return rows <= 72
        if not 3584 <= N <= 6144 or K < 4096:
            return False
        if whole or K >= 8192:
            return True
        if N <= 4096:
            return rows > 128 or K >= 6144
        if N < 5632:
            return 96 < rows < 128
        return rows <= 160 or K >= 5120
    if N > 4096:
        return False
    if K < 3072:
        return K == 2048 or (K == 1024 and not 1536 < N < 2560)
    if K > 5120:
        return rows >= 48 and (N >= 3072 or (whole and N >= 1536))
    return (N <= 2048 or (rows == 64 and K % 512 == 0)
            or (rows <= 32 and K >= 4096))


def _rows_before_rope(rows: int, N: int, K: int) -> bool:
    """As above with the rotary embedding and the cache's rows behind: 128 x 6144 x
    4096 27.1 / 28.5, 192 32.0 / 36.8, 144 29.9 / 42.4 (176 31.3 / 29.2), 128 x 7168 x
    5120 35.6 / 36.6, 192 x 10240 x 3584 37.9 / 42.0, 144 x 8192 x 8192 47.4 / 50.4;
    past the lines 96 x 4608 x 3584 23.6 / 23.4, 144 x 4608 x 4096 27.3 / 25.5, 135 x
    5376 x 4096 28.7 / 26.4, 128 x 8192 x 4096 32.5 / 30.0, 144 34.9 / 29.2, 128 x 10240
    x 3584 32.1 / 31.5.
    17 to 48 rows (decode steps of six layers 560 -> 546 and 643 -> 627), rows of W of
    2048 entries, where ranges of K fill the CUs with
    whole steps (up to 2048 rows of W, or a multiple of 1024): 17 x 2048 x 2048 10.3 /
    14.2, 17 x 3072 x 2048 12.8 / 15.2, 32 13.7 / 15.3, 48 14.7 / 15.4, 48 x 5120 x 2048
    15.5 / 16.1; past the lines 57 x 4096 x 2048 15.6 / 15.5, 45 x 2304 x 2048 17.2 /
    14.8, 47 x 3008 x 2048 16.6 / 15.2, 32 x 1536 x 1536 12.2 / 10.1, 32 x 3072 x 2304
    13.8 / 12.7, 32 x 3072 x 2560 14.3 / 13.0; 48 x 3584 x 2048 14.7 / 15.0 and 48 x 6144 x
    2048 16.6 / 16.6 are not worth a line."""
    if 17 <= rows <= 48 and K == 2048:
        return 1536 <= N <= 2048 or (N <= 5120 and N % 1024 == 0)
    if not 128 <= rows <= 192 or not 4608 <= N <= 10240 or K < 3584:
        return False
    if rows % 32 == 0:
        return N <= 6144 or K >= 5120 or (N >= 9216 and rows * K >= 1 << 19)
    if N < 5632:
        return False
    return K >= 8192 or (N <= 6144 and (rows <= 160 or K >= 5120))


def _rows_before_gate(rows: int, N: int, K: int) -> bool:
    """As above with the activation behind, in tiles that have all of K and fill
    the CUs once, rows of W a power of two apart or nearly (where the library is
    slow): 17 x 28672 x 4096 49.5 / 56.4, 64 51.7 / 55.4, 64 x 28672 x 2048 30.7 / 33.1,
    64 x 32768 x 8192 105 / 123; past the lines 96 x 28672 x 4096 59.5 / 56.3, 64 x
    24576 x 4096 50.8 / 49.0, 17 x 28672 x 2560 36.6 / 31.7, 64 x 57344 x 4096 106 /
    102; no wide tiles where N is no multiple of 128: 63 x 28224 x 4096 61.4 / 55.3."""
    return (17 <= rows <= 64 and 28160 <= N <= 32768 and N % 128 == 0
            and K % 2048 == 0)


_UNTUNED = {"": (_few_rows_alone, _long_rows),
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


def dense(*tensors) -> bool:
    """Dense tensors (or None) that may be accessed 16 bytes at a time."""
    return all(t is None or (t.is_contiguous() and t.data_ptr() % 16 == 0)
               for t in tensors)


def fused(x: torch.Tensor, w: torch.Tensor, *before) -> int:
    """What the launch of x @ w.T may have around it: 0 nothing, 1 the rotary
    embedding and the cache's rows behind it, 2 the residual's sum and the norm
    (of `before`: residual and weights) before it too. That is as many rows as
    LDS has room for (a launch of its own costs a decode step 3.5 us and up; the
    norm in every workgroup of 8 x 4096 entries as much)."""
    if x.shape[0] > 16:
        return 0
    entries = x.shape[0] * x.shape[-1]
    if (entries > _LDS_X or _choose(x, w, "around") != 1
            or not _fits(x, w) or (w.shape[0] + 32) * w.shape[1] >= 1 << 31):
        return 0
    return 2 if entries <= _LDS_NORM_X and dense(x, *before) else 1


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

    if x.dim() == 2 and fused(x, w, residual, norm_w) == 2:
        return ops.skinny_norm_gated(x, residual, norm_w, eps, w)
    add_norm = (ops.fused_add_rms_norm if x.dim() == 2
                else ops.add_rms_norm_parts)
    x, residual = add_norm(x, residual, norm_w, eps)
    return silu_mul(x, w), residual


def reset() -> None:
    _POLICY.clear()
