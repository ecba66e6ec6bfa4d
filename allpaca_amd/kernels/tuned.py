"""Checked wrappers of the bfloat16 MFMA kernels (library `tuned`).  Each checks what the kernel
assumes.  Matrix products take weights in the tiled layout (`packing.PackedWeight`), which only
matrices of a width that is a multiple of 8 get (`ops.prepare_matrix`): other widths stay row-major
and run on the plain kernel.  Attention returns False for sizes it does not take (a page size that is
no multiple of 8, a head size that is no multiple of 16 or above 256) and the caller runs the plain
kernel: never a wrong result."""
from __future__ import annotations

import functools
import math
from typing import Optional

import torch

from . import lib as _lib
from . import ops as _ops
from .packing import PackedWeight

CHIP_UNITS = 256   # compute units the rules below were measured on
MANY_ROWS_SPLIT_MAX = 1024   # up to here the tiled kernel may cut K into slices to get enough blocks
SKINNY_MAX_ROWS = 16     # the streaming kernel: up to one 16-row tile of activations
ROWS_MAX = 64            # the kernel that finishes a product of 17 rows or more in one launch (`gemm_rows_bf16.hip`)
SPLITK_MAX_ROWS = 128    # the tiled kernel with K cut into slices: 17..128 rows, where the one above does not take them


def _k_split(M: int, N: int, K: int) -> int:
    """Slices of K for the split kernel with 17..128 rows: about 240 blocks in all (measured best at the shapes of 3B
    and 8B models: 32 column tiles in 6-8 slices, 48 in 4-5, 224 whole), at least 4 K-steps of 64 each."""
    blocks = -(-N // 128) * -(-M // 128)
    s = max(1, min(12, round(240 / blocks)))
    return max(1, min(s, K // 256))


def _k_split_many_rows(M: int, N: int, K: int) -> int:
    """Slices of K on 128 x 128 tiles for 129..1024 rows: a matrix with few output columns gives the 128 x 128 tiles too few blocks
    for 256 compute units (o_proj and down of an 8B model at 512 rows: 128), and slicing K, at the price of writing
    and adding float32 partial sums, was measured faster up to about 200 blocks (down, 4096 x 14336, 256 rows: 150
    us whole, 52 us in 4 slices); with more outputs than K and 150 blocks or more it was not."""
    blocks = -(-N // 128) * -(-M // 128)
    if blocks <= 56:
        s = 5
    elif blocks <= 68:
        s = 4
    elif blocks <= 88:
        s = 3
    elif blocks <= 208 and not (blocks >= 150 and N > K):
        s = 2
    else:
        s = 1
    return max(1, min(s, K // 256))


DIRECT_SLICES_MIN_ROWS = 257   # the kernel that keeps the weights out of LDS takes slices from here on
DIRECT_MIN_ROWS = 1024         # and K in one piece whatever the columns


def _direct_slices_us(M: int, N: int, s: int) -> float:
    """Microseconds of that kernel for 4,096 columns of K a slice (`direct_slices` in `csrc/host/rules.h`)."""
    us = []
    for nf in (3, 4, 5, 6, 8):
        tiles = -(-M // 128) * -(-N // (64 * nf))
        rounds = -(-(-(-tiles // 8) * s) // (CHIP_UNITS // 8))
        us.append(rounds * (12.0 + nf * (7.5 + 3.8 * (tiles * s) / (rounds * CHIP_UNITS))))
    return min(us)


@functools.lru_cache(maxsize=4096)   # (8 us of Python a product otherwise)
def _slices_many_rows(M: int, N: int, K: int):
    """(slices of K, whether the kernel without weights in LDS takes them) for 129..1024 rows.  From 257 rows on that
    kernel's slices, which have to be of one length in pieces of 128 columns, are held against what the 128 x 128 tile
    does (its slices or K whole, `_k_split_many_rows`) by the expected microseconds: `_direct_slices_us`; two blocks of the
    tile share a unit, 27 to 40 for 256 of them and 64 for 512, up to 1.23 times that where the column tiles are no multiple of
    the 8 XCDs, which then all fetch all of W; the adding kernel 9 and 1.6 a slice and 2^20 outputs; K whole 6 more for
    what the adding kernel would have done on the way, the norm's row or the rotation.  Against 8,500 products of 257 to 1,024
    rows (K 768 to 14,336 into 640 to 11,008 columns, 900 sizes in 1 to 8 slices on either kernel) the times are off by 5 %
    (root mean square), and what is chosen takes 0.94 of the tile's time in the mean, 1.08 at worst.  K without many
    divisors stays with the tile, whose slices need none: 384 rows, K 15,104 into 640 columns 84 us in the two slices that
    the other kernel has, 33 in five.  512 rows, 4,096 x 14,336: 78 in three slices on the tile, 70 in four on the other."""
    s = _k_split_many_rows(M, N, K)
    if not (DIRECT_SLICES_MIN_ROWS <= M <= MANY_ROWS_SPLIT_MAX) or K % 128 or N % 4:
        return s, False
    outputs = M * N / 1048576.0
    tiles = -(-M // 128) * -(-N // 128)
    if M < DIRECT_MIN_ROWS and tiles <= CHIP_UNITS:
        whole = 11.0 + (30.5 + 9.0 * tiles / CHIP_UNITS) * (K / 4096.0)
    else:
        whole = 12.0 + _direct_slices_us(M, N, 1) * (K / 4096.0)
    best, direct, least = s, False, 0.96 * whole
    if s > 1:
        blocks = tiles * s
        full = (blocks - 1) // 512
        rest = blocks - 512 * full
        us = 64.5 * full + (48.7 if rest > CHIP_UNITS else 27.3) + 12.6 * (min(rest, CHIP_UNITS) / CHIP_UNITS)
        if -(-N // 128) % 8:
            us *= 1.0 + 0.23 * min(blocks, CHIP_UNITS) / CHIP_UNITS
        least = 0.96 * (us * (K / (4096.0 * s)) + 8.6 + (1.6 * s + 0.3) * outputs)
        if whole < least:
            best, least = 1, whole
    for s in (2, 3, 4, 6, 8):
        if K % (128 * s) or K < 256 * s:
            continue
        us = _direct_slices_us(M, N, s) * (K / (4096.0 * s)) + 8.0 + (1.5 * s + 0.7) * outputs
        if us < least:
            best, direct, least = s, True, us
    return best, direct


def _tiled_k_split(M: int, N: int, K: int, gated: bool = False) -> int:
    """Slices of K on the tiled kernels for M rows (1: K in one piece).  gated: gate and up in one product, N columns in all."""
    if M <= SPLITK_MAX_ROWS:
        return _k_split(M, N, K)
    if M > MANY_ROWS_SPLIT_MAX:
        return 1
    return _k_split_many_rows(M, N, K) if gated else _slices_many_rows(M, N, K)[0]


def _rows_take(a: torch.Tensor, w: PackedWeight, wu: Optional[PackedWeight], out: torch.Tensor, N: int, mode: int) -> bool:
    """Whether such a product of 17 to 64 rows runs in one launch, without slices (N: columns of each matrix)."""
    M, K = a.shape
    return bool(SKINNY_MAX_ROWS < M <= ROWS_MAX and _lib.load("tuned").apc_gemm_rows_takes(
        mode, a.data_ptr(), a.stride(0), w.data.data_ptr(), wu.data.data_ptr() if wu is not None else 0, out.data_ptr(),
        out.stride(0), M, N, K))


def _ss_parts_max(M: int) -> int:
    """Sums of x^2 a row that the products behind a norm take."""
    return 1024 if M <= ROWS_MAX else 256


# The chip these rules and the kernels' launch plans were measured on (`csrc/host/rules.h`, `gemm_direct_bf16.hip`:
# rounds of 256 blocks over 8 XCDs; `attention_wide_bf16.hip`: 160 KiB of LDS a compute unit).
CHIP_LDS_BYTES = 160 * 1024
_chips_checked: set = set()


def check_chip(device: torch.device) -> None:
    """Says so, once per device, if the GPU is not the one the dispatch rules were measured on: the results stay
    right (no kernel assumes the counts for correctness), the cuts may be badly chosen."""
    import warnings
    key = (device.type, device.index)
    if device.type != "cuda" or key in _chips_checked:
        return
    _chips_checked.add(key)
    prop = torch.cuda.get_device_properties(device)
    units = getattr(prop, "multi_processor_count", CHIP_UNITS)
    lds = getattr(prop, "shared_memory_per_block_optin", 0) or getattr(prop, "shared_memory_per_block", 0)
    if units != CHIP_UNITS or (lds and lds < CHIP_LDS_BYTES):
        warnings.warn(f"{prop.name}: {units} compute units and {lds} bytes of LDS a block; the bfloat16 kernels' dispatch "
                      f"rules were measured on {CHIP_UNITS} units with {CHIP_LDS_BYTES} bytes and may be badly tuned here")


def _aligned(*ts: torch.Tensor) -> bool:
    return all(t.data_ptr() % 16 == 0 for t in ts)


def _act_ok(a: torch.Tensor) -> bool:
    return (a.dtype == torch.bfloat16 and a.shape[1] % 8 == 0 and _ops._rows(a, "a") % 8 == 0 and _aligned(a))


MODE_ACT = 16     # the products' modes from here on: an activation (MODE_ACT + its code) on the sums, bfloat16 out


def gemm_bf16(a: torch.Tensor, w: PackedWeight, out: torch.Tensor, accumulate: bool = False, activation: int = 0) -> None:
    """out = a . w^T (bfloat16 or float32 out), or out += a . w^T (float32 out); w in the tiled layout.  `activation`
    (a code of `ops.ACTIVATIONS`): out = act(a . w^T), applied to the float32 sums, bfloat16 out."""
    _ops._gpu(a, w.data, out)
    M, K = a.shape
    N = w.N
    if not (w.K == K):
        raise ValueError(f"gemm: a is [*, {K}] but w is {w.shape}")
    if not (out.shape == (M, N)):
        raise ValueError(f"gemm: out must be [{M}, {N}], got {tuple(out.shape)}")
    _ops._need(not accumulate or out.dtype == torch.float32, "gemm: accumulation needs a float32 destination")
    _ops._need(out.dtype in (torch.bfloat16, torch.float32), "gemm: out must be bfloat16 or float32")
    _ops._need(not activation or (not accumulate and out.dtype == torch.bfloat16), "gemm: an activation stores bfloat16")
    _ops._need(w.data.is_contiguous() and w.data.shape[0] * 16 >= N and w.data.shape[1] * 32 >= K,
               "gemm: the tiled weight does not cover [N, K]")
    if not _act_ok(a):
        raise ValueError("gemm_bf16: activations must be bfloat16 rows of a width and stride that are multiples "
                         "of 8, 16-byte aligned")
    lda, ldc = _ops._rows(a, "a"), _ops._rows(out, "out")
    mode = MODE_ACT + activation if activation else 2 if accumulate else (0 if out.dtype == torch.bfloat16 else 1)
    L = _lib.load("tuned")
    if M > SKINNY_MAX_ROWS:
        # more than 1,024 rows: the product of many rows says itself whether it wants K in two slices
        ks = _tiled_k_split(M, N, K) if M <= MANY_ROWS_SPLIT_MAX else L.apc_gemm_direct_k_split(M, N, K)
        if ks > 1 and not _rows_take(a, w, None, out, N, mode):
            ws = torch.empty(ks * M * N, dtype=torch.float32, device=a.device)
            _lib.check(L.apc_gemm_splitk_bf16(a.data_ptr(), lda, w.data.data_ptr(), 0, out.data_ptr(), ldc, M, N, K,
                                              mode, ks, ws.data_ptr(), _ops._stream()), "gemm_splitk_bf16")
            return
    fn = L.apc_skinny_gemm_bf16 if M <= SKINNY_MAX_ROWS else L.apc_gemm_bf16
    _lib.check(fn(a.data_ptr(), lda, w.data.data_ptr(), out.data_ptr(), ldc, M, N, K, mode, _ops._stream()),
               "gemm_bf16")


def swiglu_bf16(h: torch.Tensor, wg: PackedWeight, wu: PackedWeight, out: torch.Tensor) -> None:
    """out[t, f] = silu(h . Wg[f]) * (h . Wu[f]); Wg, Wu in the tiled layout."""
    _ops._gpu(h, wg.data, wu.data, out)
    M, K = h.shape
    F = out.shape[1]
    if not (wg.shape == (F, K) and wu.shape == (F, K)):
        raise ValueError(f"swiglu: weights must both be [{F}, {K}]")
    _ops._need(out.shape[0] == M and out.dtype == torch.bfloat16, "swiglu: out must be bfloat16 [rows, F]")
    if not _act_ok(h):
        raise ValueError("swiglu_bf16: activations must be bfloat16 rows of a width and stride that are multiples "
                         "of 8, 16-byte aligned")
    lda, ldc = _ops._rows(h, "h"), _ops._rows(out, "out")
    L = _lib.load("tuned")
    ks = _tiled_k_split(M, 2 * F, K, True) if M > SKINNY_MAX_ROWS else 1
    if ks > 1 and not _rows_take(h, wg, wu, out, F, 3):
        ws = torch.empty(2 * ks * M * F, dtype=torch.float32, device=h.device)
        _lib.check(L.apc_gemm_splitk_bf16(h.data_ptr(), lda, wg.data.data_ptr(), wu.data.data_ptr(), out.data_ptr(), ldc,
                                          M, F, K, 3, ks, ws.data_ptr(), _ops._stream()), "gemm_splitk_bf16")
        return
    fn = L.apc_skinny_swiglu_bf16 if M <= SKINNY_MAX_ROWS else L.apc_gemm_swiglu_bf16
    _lib.check(fn(h.data_ptr(), lda, wg.data.data_ptr(), wu.data.data_ptr(), out.data_ptr(), ldc, M, F, K,
                  _ops._stream()), "swiglu_bf16")


def gemm_emit_bf16(a: torch.Tensor, w: PackedWeight, residual: torch.Tensor, g: torch.Tensor):
    """residual += a . w^T, and for the RMS norm with weight g that reads the residual next: the row
    bfloat16(residual * g) and sums of residual^2 per row and group of columns.  Returns (raw [M, N], ss) or None,
    with nothing done, for sizes no kernel takes.  ss is [16, ceil(N/16) rounded up to 4] from the streaming kernel
    (up to 16 rows), [M, N/16] from the kernel of up to 64 rows and [M, ceil(N/256)] from the tiled kernel with K in
    slices; the products below take what the same number of rows gives."""
    _ops._gpu(a, w.data, residual, g)
    M, K = a.shape
    N = w.N
    if (not _act_ok(a) or residual.dtype != torch.float32 or g.dtype != torch.float32 or g.numel() != N
            or not g.is_contiguous()):
        return None
    if not (w.K == K and residual.shape == (M, N)):
        raise ValueError(f"gemm: a [{M}, {K}], w {w.shape}, residual {tuple(residual.shape)}")
    L = _lib.load("tuned")
    lda, ldc = _ops._rows(a, "a"), _ops._rows(residual, "residual")
    if M > MANY_ROWS_SPLIT_MAX:
        # the product of many rows: its own epilogue leaves the row, or with K in two slices the kernel that adds them
        # (sums of squares per tile of columns, or per 1,024 columns)
        parts = L.apc_gemm_direct_emit_parts(a.data_ptr(), lda, residual.data_ptr(), ldc, M, N, K)
        if not parts:
            return None
        raw = torch.empty((M, N), dtype=torch.bfloat16, device=a.device)
        ss = torch.empty((M, parts), dtype=torch.float32, device=a.device)
        ks = L.apc_gemm_direct_emit_k_split(M, N, K)
        ws = torch.empty(ks * M * N, dtype=torch.float32, device=a.device) if ks > 1 else None
        _lib.check(L.apc_gemm_direct_emit_bf16(a.data_ptr(), lda, w.data.data_ptr(), residual.data_ptr(), ldc, M, N, K,
                                               g.data_ptr(), raw.data_ptr(), N, ss.data_ptr(), parts,
                                               ws.data_ptr() if ws is not None else 0, _ops._stream()),
                   "gemm_direct_emit_bf16")
        return raw, ss
    if SKINNY_MAX_ROWS < M <= ROWS_MAX and N // 16 <= _ss_parts_max(M) and L.apc_gemm_rows_emit_takes(
            a.data_ptr(), lda, w.data.data_ptr(), residual.data_ptr(), ldc, M, N, K, g.data_ptr()):
        raw = torch.empty((M, N), dtype=torch.bfloat16, device=a.device)
        ss = torch.empty((M, N // 16), dtype=torch.float32, device=a.device)
        _lib.check(L.apc_gemm_rows_emit_bf16(a.data_ptr(), lda, w.data.data_ptr(), residual.data_ptr(), ldc, M, N, K,
                                             g.data_ptr(), raw.data_ptr(), N, ss.data_ptr(), _ops._stream()),
                   "gemm_rows_emit_bf16")
        return raw, ss
    if M > SKINNY_MAX_ROWS:   # the tiled kernel: only where K is cut into slices (the finishing kernel leaves the row)
        ks = _tiled_k_split(M, N, K)
        if ks == 1:
            # With K in one piece the product's own epilogue would have to do it; measured at 2,048 rows that costs
            # 20-27 us a product, more than the norm's kernel (10 us) that it would save.
            return None
        raw = torch.empty((M, N), dtype=torch.bfloat16, device=a.device)
        ss = torch.empty((M, -(-N // 256)), dtype=torch.float32, device=a.device)
        ws = torch.empty(ks * M * N, dtype=torch.float32, device=a.device)
        _lib.check(L.apc_gemm_splitk_emit_bf16(a.data_ptr(), lda, w.data.data_ptr(), residual.data_ptr(), ldc, M, N, K,
                                               ks, ws.data_ptr(), g.data_ptr(), raw.data_ptr(), N, ss.data_ptr(),
                                               _ops._stream()), "gemm_splitk_emit_bf16")
        return raw, ss
    raw = torch.empty((M, N), dtype=torch.bfloat16, device=a.device)
    ss = torch.empty((16, -(-(-(-N // 16)) // 4) * 4), dtype=torch.float32, device=a.device)
    _lib.check(L.apc_skinny_gemm_emit_bf16(a.data_ptr(), lda, w.data.data_ptr(), residual.data_ptr(), ldc, M, N, K,
                                           g.data_ptr(), raw.data_ptr(), N, ss.data_ptr(), _ops._stream()),
               "skinny_gemm_emit_bf16")
    return raw, ss


def _pre_ok(raw: torch.Tensor, ss: torch.Tensor, K: int) -> bool:
    return (raw.shape[0] <= SKINNY_MAX_ROWS and _act_ok(raw) and ss.dtype == torch.float32 and ss.is_contiguous()
            and tuple(ss.shape) == (16, -(-(-(-K // 16)) // 4) * 4))


def _pre_tiled(raw: torch.Tensor, ss: torch.Tensor, eps: float, w, wu, out: torch.Tensor, n_cols: int, mode: int) -> bool:
    """The same with more than 16 rows, in one launch or on the tiled kernel, K in slices or in one piece: ss is [M,
    parts] with up to 256 sums of squares a row (what the tiled kernels leave: a part per 256 or per 128 columns), up to 64
    rows 1,024 (a part per 16 columns)."""
    M, K = raw.shape
    if not (M > SKINNY_MAX_ROWS and _act_ok(raw) and ss.dtype == torch.float32 and ss.is_contiguous()
            and ss.dim() == 2 and ss.shape[0] == M and 1 <= ss.shape[1] <= _ss_parts_max(M)):
        return False
    n_mats = 2 if wu is not None else 1
    ks = _tiled_k_split(M, n_cols * n_mats, K, wu is not None)
    L = _lib.load("tuned")
    wu_ptr = wu.data.data_ptr() if wu is not None else 0
    if ks == 1 or _rows_take(raw, w, wu, out, n_cols, mode):
        _lib.check(L.apc_gemm_pre_bf16(raw.data_ptr(), _ops._rows(raw, "raw"), ss.data_ptr(), ss.shape[1], float(eps),
                                       w.data.data_ptr(), wu_ptr, out.data_ptr(), _ops._rows(out, "out"), M, n_cols, K,
                                       mode, _ops._stream()), "gemm_pre_bf16")
        return True
    ws = torch.empty(n_mats * ks * M * n_cols, dtype=torch.float32, device=raw.device)
    _lib.check(L.apc_gemm_splitk_pre_bf16(raw.data_ptr(), _ops._rows(raw, "raw"), ss.data_ptr(), ss.shape[1], float(eps),
                                          w.data.data_ptr(), wu_ptr, out.data_ptr(), _ops._rows(out, "out"), M, n_cols,
                                          K, mode, ks, ws.data_ptr(), _ops._stream()), "gemm_splitk_pre_bf16")
    return True


def gemm_pre_bf16(raw: torch.Tensor, ss: torch.Tensor, eps: float, w: PackedWeight, out: torch.Tensor) -> bool:
    """out = (raw . w^T) / sqrt(sum(ss) / K + eps) for a row that `gemm_emit_bf16` left: the product of the
    normalised row.  False, with nothing done, for sizes the kernel does not take."""
    _ops._gpu(raw, ss, w.data, out)
    M, K = raw.shape
    if out.dtype not in (torch.bfloat16, torch.float32):
        return False
    if not (w.K == K and out.shape == (M, w.N)):
        raise ValueError(f"gemm: raw [{M}, {K}], w {w.shape}, out {tuple(out.shape)}")
    if M > SKINNY_MAX_ROWS:
        return _pre_tiled(raw, ss, eps, w, None, out, w.N, 0 if out.dtype == torch.bfloat16 else 1)
    if not _pre_ok(raw, ss, K):
        return False
    L = _lib.load("tuned")
    _lib.check(L.apc_skinny_gemm_pre_bf16(raw.data_ptr(), _ops._rows(raw, "raw"), ss.data_ptr(), -(-K // 16), float(eps),
                                          w.data.data_ptr(), out.data_ptr(), _ops._rows(out, "out"), M, w.N, K,
                                          0 if out.dtype == torch.bfloat16 else 1, _ops._stream()),
               "skinny_gemm_pre_bf16")
    return True


def qkv_rope_bf16(a: torch.Tensor, pre, w: PackedWeight, q_out: torch.Tensor, n_heads: int, n_kv_heads: int,
                  head_dim: int, cos_sin: torch.Tensor, positions: torch.Tensor, row_seg: torch.Tensor,
                  block_table: torch.Tensor, cache: torch.Tensor, page_tokens: int) -> bool:
    """q, k, v in one product that also rotates q and k (whole heads) and writes k and v into the pages; rotated q
    goes to the first n_heads * head_dim columns of q_out.  Up to 16 rows: the streaming kernel (head size a
    multiple of 32); up to 64 the kernel that finishes in one launch, where that is faster; more rows: the tiled kernel
    where it cuts K into slices, in its finishing kernel (256 a multiple of the head size), and the kernel whose weights go
    straight into registers where that takes the product in one piece (heads of 64 and 128).  `a`: the normalised rows, or with `pre` = (ss, eps) the row that
    `gemm_emit_bf16` left.  False, with nothing done, for sizes neither takes."""
    _ops._gpu(a, w.data, q_out, cos_sin, positions, row_seg, block_table, cache)
    M, K = a.shape
    H, Hk, d = n_heads, n_kv_heads, head_dim
    N = (H + 2 * Hk) * d
    few = M <= SKINNY_MAX_ROWS
    if not (_act_ok(a) and q_out.dtype == torch.bfloat16 and cache.dtype == torch.bfloat16):
        return False
    if few and not (d % 32 == 0 and q_out.stride(0) % 4 == 0 and q_out.data_ptr() % 8 == 0):
        return False
    ks = 1 if few else _tiled_k_split(M, N, K)
    rows = SKINNY_MAX_ROWS < M <= ROWS_MAX and _lib.load("tuned").apc_gemm_rows_qkv_takes(
        a.data_ptr(), a.stride(0), w.data.data_ptr(), q_out.data_ptr(), q_out.stride(0), M, K, H, Hk, d, cos_sin.data_ptr(),
        cache.data_ptr())
    direct = not few and ks == 1 and not rows and _lib.load("tuned").apc_gemm_direct_qkv_takes(
        a.data_ptr(), a.stride(0), q_out.data_ptr(), q_out.stride(0), M, K, H, Hk, d, cos_sin.data_ptr(), cache.data_ptr())
    if not few and not direct and ((ks == 1 and not rows) or 256 % d or d % 2):
        return False
    ss, eps = None, 0.0
    if pre is not None:
        ss, eps = pre
        if few and not _pre_ok(a, ss, K):
            return False
        if not few and not (ss.dtype == torch.float32 and ss.is_contiguous() and ss.dim() == 2 and ss.shape[0] == M
                            and 1 <= ss.shape[1] and (direct or ss.shape[1] <= _ss_parts_max(M))):
            return False
    if not (w.K == K and w.N == N and q_out.shape[0] == M and q_out.shape[1] >= H * d):
        raise ValueError(f"qkv: a [{M}, {K}], w {w.shape}, {H}+2*{Hk} heads of {d}, q_out {tuple(q_out.shape)}")
    _ops._need(cos_sin.dtype == torch.float32 and cos_sin.is_contiguous() and tuple(cos_sin.shape[1:]) == (2, d // 2),
               "cos/sin table must be float32 [positions, 2, head_dim/2]")
    if not (cache.dim() == 5 and cache.is_contiguous() and tuple(cache.shape[1:]) == (2, Hk, page_tokens, d)):
        raise ValueError(f"cache must be [pages, 2, {Hk}, {page_tokens}, {d}], got {tuple(cache.shape)}")
    _ops._need(block_table.dim() == 2 and block_table.dtype == torch.int32 and block_table.is_contiguous(),
               "block table must be contiguous int32 [segments, blocks]")
    L = _lib.load("tuned")
    ss_ptr = ss.data_ptr() if ss is not None else 0
    if few:
        _lib.check(L.apc_skinny_qkv_rope_bf16(
            a.data_ptr(), _ops._rows(a, "a"), ss_ptr, -(-K // 16) if ss is not None else 0, float(eps), w.data.data_ptr(),
            q_out.data_ptr(), _ops._rows(q_out, "q_out"), M, K, H, Hk, d, cos_sin.data_ptr(),
            _ops._i32(positions, M, "positions"), _ops._i32(row_seg, M, "row_seg"), block_table.data_ptr(),
            block_table.shape[1], cache.data_ptr(), page_tokens, _ops._stream()), "skinny_qkv_rope_bf16")
        return True
    if direct:
        _lib.check(L.apc_gemm_direct_qkv_rope_bf16(
            a.data_ptr(), _ops._rows(a, "a"), ss_ptr, ss.shape[1] if ss is not None else 0, float(eps), w.data.data_ptr(),
            q_out.data_ptr(), _ops._rows(q_out, "q_out"), M, K, H, Hk, d, cos_sin.data_ptr(),
            _ops._i32(positions, M, "positions"), _ops._i32(row_seg, M, "row_seg"), block_table.data_ptr(),
            block_table.shape[1], cache.data_ptr(), page_tokens, _ops._stream()), "gemm_direct_qkv_rope_bf16")
        return True
    ws = None if rows else torch.empty(ks * M * N, dtype=torch.float32, device=a.device)
    _lib.check(L.apc_gemm_splitk_qkv_rope_bf16(
        a.data_ptr(), _ops._rows(a, "a"), ss_ptr, ss.shape[1] if ss is not None else 0, float(eps), w.data.data_ptr(),
        q_out.data_ptr(), _ops._rows(q_out, "q_out"), M, K, H, Hk, d, cos_sin.data_ptr(),
        _ops._i32(positions, M, "positions"), _ops._i32(row_seg, M, "row_seg"), block_table.data_ptr(),
        block_table.shape[1], cache.data_ptr(), page_tokens, ks, ws.data_ptr() if ws is not None else 0, _ops._stream()),
        "gemm_splitk_qkv_rope_bf16")
    return True


def swiglu_pre_bf16(raw: torch.Tensor, ss: torch.Tensor, eps: float, wg: PackedWeight, wu: PackedWeight,
                    out: torch.Tensor) -> bool:
    """SwiGLU of the normalised row, from what `gemm_emit_bf16` left (see `gemm_pre_bf16`)."""
    _ops._gpu(raw, ss, wg.data, wu.data, out)
    M, K = raw.shape
    F = out.shape[1]
    if out.dtype != torch.bfloat16:
        return False
    if not (wg.shape == (F, K) and wu.shape == (F, K) and out.shape[0] == M):
        raise ValueError(f"swiglu: weights must both be [{F}, {K}]")
    if M > SKINNY_MAX_ROWS:
        return _pre_tiled(raw, ss, eps, wg, wu, out, F, 3)
    if not _pre_ok(raw, ss, K):
        return False
    L = _lib.load("tuned")
    _lib.check(L.apc_skinny_swiglu_pre_bf16(raw.data_ptr(), _ops._rows(raw, "raw"), ss.data_ptr(), -(-K // 16),
                                            float(eps), wg.data.data_ptr(), wu.data.data_ptr(), out.data_ptr(),
                                            _ops._rows(out, "out"), M, F, K, _ops._stream()), "skinny_swiglu_pre_bf16")
    return True


def _decode_parts(pairs: int, span: int) -> int:
    """Ranges that the decode kernel cuts the keys of every row into (four to a block, one per wave): as many blocks
    a (row, kv head) pair as keep the launch at one block a compute unit or under, and no range under 64 keys.  The
    kernel sizes a row's ranges from the row's own length, so the count depends on the step's shape alone.  Measured at
    8B shapes (32 heads over 8, heads of 128), 1 to 16 rows over 512 to 8,192 keys, ranges of 64 to 512 keys: the
    fastest choice was in every case the shortest range whose launch fits the chip once (8 rows over 2,063 keys: 256
    blocks 18.9 us, 320 blocks 21.4 us, 192 blocks 20.6 us; over 8,192 keys: 256 blocks 53.3 us, 512 blocks 54.6 us,
    1,024 blocks 56.5 us)."""
    per_pair = max(1, CHIP_UNITS // max(1, pairs))
    return max(1, min(WHOLE_WAVES * per_pair, -(-span // 64)))


# Keys of a range of the decode kernel, the same for every row and counted from position 0, instead of the rule above
# (0: the rule): for measurements and tests.
KEYS_PER_PART = 0


# From how many (row, kv head) pairs on a decode step's attention runs as one block per pair that finishes its heads
# itself (no partial results through memory, no second kernel): the pairs alone then give every compute unit work
# (measured at the shapes of an 8B model: 7-15 % faster from 32 rows on, slower with 16).
WHOLE_MIN_PAIRS = 256
WHOLE_WAVES = 4   # waves of such a block (NW in attention_bf16.hip)


# From so many pairs on, in steps whose longest row may have more keys than this, the rows' work may be dealt out evenly over
# all waves of one round of blocks (DEC_EVEN in attention_bf16.hip) instead of a block a pair, whose longest row sets the
# launch's time; whether it is, the rows' lengths say (`_even_pays`).  With fewer pairs the way below, which cuts every pair
# for itself, is faster (16 rows of 2,048 26.8 / 30 us, 8 rows 17.6 / 26).  Where a block has no room for a pair (16 heads of
# 256 on a kv head) a pair's keys go to parts in memory: from 1,024 pairs on shares are faster whatever the lengths (1,024
# rows of 1,100 250 / 205, of 30 to 1,100 125 / 115), with 256 pairs not (61 / 92, 47 / 62).  More pairs than the compiled
# executor has counters for keep a block each.
EVEN_MIN_PAIRS, EVEN_MIN_SPAN = 256, 1024
EVEN_MAX_PAIRS, EVEN_ALONE_MIN_PAIRS = 4096, 1024


def _decode_even(pairs: int, span: int, pair_fits: bool = True) -> bool:
    least = EVEN_MIN_PAIRS if pair_fits else max(EVEN_MIN_PAIRS, EVEN_ALONE_MIN_PAIRS)
    return least <= pairs <= EVEN_MAX_PAIRS and span > EVEN_MIN_SPAN


def _even_pays(steps: int, longest: int, n_rows: int, tiles: int, window: int) -> bool:
    """Whether shares beat a block a pair for the lengths at hand (`StepInfo.decode_work`, which a window cuts), by the time
    of either in units of a wave's step of 32 keys.  Shares: a wave's share, a few units for the pieces' way through memory,
    and a look at all rows.  A block a pair: the same work, or the longest row's chain over four waves, slowed by the blocks
    that share its compute unit.  Fitted to 774 launches (1 to 32 kv heads of 64 to 256, 8 to 512 rows of equal, spread and
    single long lengths) of the kernels before keys came in whole lines, when the choice was on average 0.5 % over the better
    of the two.  Since then both are faster, a block a pair by more where two share a unit: of 684 launches (1 to 16 kv heads and
    32) the choice is 0.9 % over the better one in the mean and 18 % at worst (512 rows of 500 to 1,500 keys on one kv head 49 / 58
    us); shares alone are 2.9 %, a block a pair alone 37 %.  Microseconds a layer, block a pair / shares, 8 kv heads of 128: 32 rows
    of 1,100 keys 27.1 / 32.5, of 2,048 46.1 / 52.6, of 1,000 to 2,048 37.3 / 40.2, of 90 to 2,100 28.5 / 23.5; 64 rows of 1,100 50.5 /
    56.2, of 2,048 90.0 / 94.0, of 1,000 to 2,048 74.8 / 74.2, of 90 to 2,100 53.7 / 36.6, one of 8,000 beside 63 of 100 168 / 27; 128
    rows of 2,048 169.7 / 169.0.  32 kv heads of 128: 8 rows of 2,048 45.5 / 51.4, of 90 to 2,100 23.0 / 22.9, 16 rows of those 46 / 31."""
    if window:
        most = window // 32 + 1
        longest, steps = min(longest, most), min(steps, n_rows * most)
    waves = max(1, CHIP_UNITS // tiles) * WHOLE_WAVES
    units, share = n_rows * WHOLE_WAVES / waves, (steps + 2 * n_rows) / waves
    whole = max(1.03 * share + 2.5 + 1.1 * units, 4.1 + 0.245 * longest * min(math.ceil(units), 2.8))
    return 7.3 + max(share, 8.3) + 0.05 * (n_rows / 64) < whole


def decode_shape(n_heads: int, n_kv_heads: int, head_dim: int, window: int) -> tuple:
    """What the way of a layer's decoded rows depends on beside the rows: (tiles of heads a row, whether a block has room
    for a (row, kv head) pair, window)."""
    fits = bool(_lib.load("tuned").apc_attention_decode_whole_fits(n_heads, n_kv_heads, head_dim))
    return n_kv_heads * -(-(n_heads // n_kv_heads) // 16), fits, int(window)


def _decode_shares(rows: int, span: int, work, shape) -> bool:
    """Whether the rows of such a layer share out their work; `work`: `StepInfo.decode_work`."""
    tiles, fits, window = shape
    return (_decode_even(rows * tiles, min(span, window) if window else span, fits)
            and (not fits or _even_pays(work[0], work[1], rows, tiles, window)))


def decode_routes_differ(rows: int, span: int, shapes) -> bool:
    """Whether the rows' lengths say how some layer of these shapes divides its decoded rows."""
    return any(f and _decode_even(rows * t, min(span, w) if w else span) for t, f, w in shapes)


def decode_routes(rows: int, span: int, work, shapes) -> tuple:
    """How every one of the layers' shapes divides decoded rows of such lengths."""
    return tuple(_decode_shares(rows, span, work, s) for s in sorted(shapes))


# With fewer pairs: the blocks of a pair leave one partial result each and the one that finishes last adds them (no
# second kernel), where the sizes allow; False: partial results per wave and a kernel that merges them.
LAST_BLOCK_MERGES = True
# Portions whose tiles of 128 rows are mostly whole (heads of 128 or 64, pages of a power of two from 16 on) run on the kernel
# that takes such a tile a block (attention_wide_bf16.hip); False sends every portion to the kernels of 64-row blocks.
WIDE_TILES = True
_counters: dict = {}
# Ranges that the keys of a tile of prompt rows are cut into: never more (0 sends a tile's keys to one block always),
# and the keys a range must keep
KEY_SPLITS_MAX = 8
KEY_RANGE_MIN = 2048


def _key_splits(step, n_heads: int, window: int) -> int:
    """Into how many ranges of keys the 128-row attention kernel cuts every tile of this step: a block per (tile, head)
    leaves compute units idle when a step has few tiles (a chunk of 512 prompt tokens at 32 heads: 128 blocks for 256
    units), so the keys are shared out until the chip has a block a unit, as long as a range keeps KEY_RANGE_MIN keys
    (measured at 8B shapes, 512 rows: 1.2 times as fast at 4,096 keys, 1.56 at 32,768, a loss at 2,048: a block's
    start and the kernel that adds the ranges cost a few tiles of 64 keys), or half as many while the chip stays at
    most half full (a block alone on its compute unit and its neighbours' runs at the pace of its own chain of loads:
    128 rows over 2,048 keys in 2 ranges 1.27 times as fast, over 4,096 keys in 4 ranges 1.9 times).  1: no cutting."""
    blocks = step.n_tiles * n_heads
    pos0 = getattr(step, "host_pos0", None)
    rows = getattr(step, "host_rows", None)
    if not KEY_SPLITS_MAX or blocks <= 0 or not pos0 or not rows:
        return 1
    keys = max([p + n for p, n in zip(pos0, rows) if n > 1] or [0])     # of the longest prompt in the step
    if window:
        keys = min(keys, window + 128)
    few = min(keys // max(1, KEY_RANGE_MIN // 2), 128 // blocks)
    return max(1, min(KEY_SPLITS_MAX, 256 // blocks, max(keys // KEY_RANGE_MIN, few)))


# Bytes that partial results of such ranges may take (the engine keeps 1 GiB beside its cache for what a step needs over
# its activations); a step of many rows has blocks enough.
KEY_PARTS_MAX = 256 << 20


def _prompt_passes(pos0, rows) -> int:
    """Passes of 64 keys that the 128-row attention kernel makes over the tiles of all segments of several rows."""
    return sum((p + min(i + 128, n) - 1) // 64 + 1 for p, n in zip(pos0 or (), rows or ()) if n > 1 for i in range(0, n, 128))


def _key_splits_by_time(n_tiles: int, rows: int, n_heads: int, head_dim: int, passes: int, window: int) -> int:
    """The ranges of keys with the least time by this model (microseconds): a compute unit's blocks one after the other, a
    block 12.5 + 0.8 a pass of 64 keys; with heads of 64, where two share a unit, two together 6 + 1.15 a pass and one by
    itself 6 + 0.66; and for the kernel that adds the ranges 12 (heads of 64: 5) and its bytes at 6 TB/s.  It takes
    launches of more blocks than units, whose last round may be nearly empty, and all with heads of 64: 1,500 rows over
    24,000 keys at 32 heads of 64 (384 blocks, one and a half a unit) 459 us whole, 402, 389, 355, 367 us in 2 to 5 ranges
    (chosen: 4); over 4,000 keys 100, 96, 105, 105 (1); 700 rows over 8,000 95, 88, 92, 79, 84 (4); 300 rows over 16,000
    166, 94, 100, 82, 73 (5); 1,024 rows over 16,000 186, 172, 172, 173 (2); 1,500 rows over 16,000 at 24 heads of 128 (288
    blocks) 468, 396, 379, 376, 379 (3), over 3,000 119, 127, 135 (1); 2,048 rows over 8,000 at 32 heads 309, 346 (1).
    The ranges' partial results stay within KEY_PARTS_MAX bytes."""
    blocks = n_tiles * n_heads
    mean = passes / n_tiles
    if window:
        mean = min(mean, float(-(-window // 64) + 2))
    best, best_us = 1, 1e30
    for s in range(1, max(1, KEY_SPLITS_MAX) + 1):
        if s > 1 and s * rows * n_heads * (head_dim + 2) * 4.0 > KEY_PARTS_MAX:
            break
        unit = -(-blocks * s // CHIP_UNITS)     # blocks of the busiest compute unit
        q = mean / s
        if head_dim <= 64:
            us = (unit // 2) * (6.0 + 1.15 * q) + (unit % 2) * (6.0 + 0.66 * q)
        else:
            us = unit * (12.5 + 0.8 * q)
        if s > 1:
            us += (5.0 if head_dim <= 64 else 12.0) + s * rows * n_heads * (head_dim + 2) * 8.0 / 6e6
        if s == 1:
            best_us = 0.97 * us                 # (cut only where it is worth something)
        elif us < best_us:
            best, best_us = s, us
    return best


def _prompt_ranges(step, rows: int, n_heads: int, head_dim: int, window: int) -> int:
    """Ranges that the kernel of 128-row blocks cuts the keys of a step's tiles (`rows` rows in all) into."""
    if head_dim <= 64 or step.n_tiles * n_heads > CHIP_UNITS:
        passes = _prompt_passes(getattr(step, "host_pos0", None), getattr(step, "host_rows", None))
        return _key_splits_by_time(step.n_tiles, rows, n_heads, head_dim, passes, window)
    return _key_splits(step, n_heads, window)


def _pair_counters(device: torch.device, pairs: int, own: Optional[list] = None) -> torch.Tensor:
    """Zeroed int32 counters, one per (row, kv head tile): a call leaves them zero again, so launches that share them must
    not overlap.  `own`: the list of an engine that records its steps (`StepInfo.pair_counters`); its steps never overlap,
    and a replayed graph keeps pointing at what its recording found there.  Without it every stream has a set that lives
    as long as the process.  Grown by allocating anew; the old ones stay (graphs).  A recording that finds none large
    enough takes counters of its own, which every replay clears: what is allocated while recording is cleared by that one
    graph alone, and must not be kept for others."""
    recording = torch.cuda.is_current_stream_capturing()
    if own is None and not recording:
        own = _counters.setdefault((device.type, device.index if device.index is not None else torch.cuda.current_device(),
                                    _ops._stream()), [])
    if own and own[-1].numel() >= pairs:
        return own[-1]
    if recording:
        return torch.zeros(pairs, dtype=torch.int32, device=device)
    own.append(torch.zeros(max(1024, pairs), dtype=torch.int32, device=device))
    return own[-1]


def attention_bf16(q: torch.Tensor, q_off: int, out: torch.Tensor, n_heads: int, n_kv_heads: int, head_dim: int,
                   cache: torch.Tensor, page_tokens: int, block_table: torch.Tensor, step, window: int = 0,
                   scale: Optional[float] = None) -> bool:
    """Attention of a whole step: single-row segments on the split-key decode kernel, longer segments on the
    tiled prefill kernel (the compiled executor runs both in one launch, `apc_attention_mixed_bf16`, where the sizes allow it: the
    same bits).  Returns False (nothing done) if the sizes are not ones these kernels take."""
    _ops._gpu(q, out, cache, block_table)
    ldq, ldo = _ops._rows(q, "attention q"), _ops._rows(out, "attention out")
    T = q.shape[0]
    if scale is not None and not scale > 0:
        return False
    if (head_dim % 16 or head_dim > 256 or page_tokens % 8 or ldq % 8 or q_off % 8 or not _aligned(q, cache)
            or q.dtype != torch.bfloat16 or cache.dtype != torch.bfloat16 or out.dtype != torch.bfloat16):
        return False
    _ops._need(q_off + n_heads * head_dim <= q.shape[1], "attention: q heads exceed the row")
    _ops._need(out.shape == (T, n_heads * head_dim), "attention out must be [rows, heads*head_dim]")
    _ops._need(n_heads % n_kv_heads == 0, "heads must be a multiple of kv heads")
    if not (cache.dim() == 5 and cache.is_contiguous()
            and tuple(cache.shape[1:]) == (2, n_kv_heads, page_tokens, head_dim)):
        raise ValueError(f"cache must be [pages, 2, {n_kv_heads}, {page_tokens}, {head_dim}], got {tuple(cache.shape)}")
    _ops._need(block_table.dim() == 2 and block_table.dtype == torch.int32 and block_table.is_contiguous(),
               "block table must be contiguous int32 [segments, blocks]")
    _ops._need(step.positions.numel() >= T and step.row_seg.numel() >= T, "step rows differ from q rows")
    sc = (1.0 / math.sqrt(head_dim)) if scale is None else float(scale)
    L = _lib.load("tuned")
    stream = _ops._stream()
    shape = decode_shape(n_heads, n_kv_heads, head_dim, window)
    if getattr(step, "decode_shapes", None) is not None:
        step.decode_shapes.add(shape)
    if step.n_tiles:
        # (only the kernel of 128-row blocks cuts keys into ranges: no room is taken for the others)
        wide = WIDE_TILES and L.apc_attention_prefill_wide_takes(n_kv_heads, head_dim, page_tokens, step.n_tiles, T - step.n_decode_rows)
        splits = _prompt_ranges(step, T - step.n_decode_rows, n_heads, head_dim, int(window)) if wide else 1
        parts = (torch.empty(splits * T * n_heads * (head_dim + 2), dtype=torch.float32, device=q.device)
                 if splits > 1 else None)
        _lib.check(L.apc_attention_prefill_bf16(
            q.data_ptr(), ldq, q_off, out.data_ptr(), ldo, n_heads, n_kv_heads, head_dim, cache.data_ptr(),
            page_tokens, block_table.data_ptr(), block_table.shape[1], step.positions.data_ptr(),
            step.row_seg.data_ptr(), step.tile_row0.data_ptr(), step.tile_rows.data_ptr(), step.n_tiles,
            (T - step.n_decode_rows) if WIDE_TILES else 0, int(window), sc, splits, T,
            parts.data_ptr() if parts is not None else 0, stream), "attention_prefill_bf16")
    if step.n_decode_rows:
        n = step.n_decode_rows
        span = min(step.max_decode_context, window) if window else step.max_decode_context
        rows = step.decode_rows.data_ptr() if step.decode_rows is not None else 0
        pairs = n * n_kv_heads * -(-(n_heads // n_kv_heads) // 16)
        counters = lambda: _pair_counters(q.device, pairs, getattr(step, "pair_counters", None))  # noqa: E731
        n_parts = -(-step.max_decode_context // KEYS_PER_PART) if KEYS_PER_PART else _decode_parts(pairs, span)
        pair_fits = shape[1]
        if _decode_shares(n, step.max_decode_context, getattr(step, "decode_work", (0, 0)), shape) and not KEYS_PER_PART and ldo % 4 == 0 and out.data_ptr() % 8 == 0:
            ws = torch.empty(L.apc_attention_decode_even_workspace(n_heads, n_kv_heads, head_dim), dtype=torch.float32,
                             device=q.device)
            _lib.check(L.apc_attention_decode_even_bf16(
                q.data_ptr(), ldq, q_off, out.data_ptr(), ldo, n, n_heads, n_kv_heads, head_dim, cache.data_ptr(),
                page_tokens, block_table.data_ptr(), block_table.shape[1], step.positions.data_ptr(),
                step.row_seg.data_ptr(), rows, int(window), sc, ws.data_ptr(),
                counters().data_ptr(), stream), "attention_decode_bf16 (even shares)")
            return True
        # (rows so short that one block's waves take a pair's ranges need no partial results either)
        if (pairs >= WHOLE_MIN_PAIRS or n_parts <= WHOLE_WAVES) and pair_fits:
            _lib.check(L.apc_attention_decode_bf16(
                q.data_ptr(), ldq, q_off, out.data_ptr(), ldo, n, n_heads, n_kv_heads, head_dim, cache.data_ptr(),
                page_tokens, block_table.data_ptr(), block_table.shape[1], step.positions.data_ptr(),
                step.row_seg.data_ptr(), rows, int(window), sc, 0, 0, 0, 0, stream), "attention_decode_bf16 (whole)")
            return True
        kw = KEYS_PER_PART
        if LAST_BLOCK_MERGES and L.apc_attention_decode_last_fits(n_heads, n_kv_heads, head_dim, n_parts):
            # one partial result a block; the block of a (row, kv head) that finishes last adds them: one launch
            nz = -(-n_parts // WHOLE_WAVES)
            ws = torch.empty(n * n_heads * nz * (head_dim + 2), dtype=torch.float32, device=q.device)
            _lib.check(L.apc_attention_decode_bf16(
                q.data_ptr(), ldq, q_off, out.data_ptr(), ldo, n, n_heads, n_kv_heads, head_dim, cache.data_ptr(),
                page_tokens, block_table.data_ptr(), block_table.shape[1], step.positions.data_ptr(),
                step.row_seg.data_ptr(), rows, int(window), sc, kw, n_parts, ws.data_ptr(),
                counters().data_ptr(), stream), "attention_decode_bf16 (last block merges)")
            return True
        ws = torch.empty(n * n_heads * n_parts * (head_dim + 2), dtype=torch.float32, device=q.device)
        _lib.check(L.apc_attention_decode_bf16(
            q.data_ptr(), ldq, q_off, out.data_ptr(), ldo, n, n_heads, n_kv_heads, head_dim, cache.data_ptr(),
            page_tokens, block_table.data_ptr(), block_table.shape[1], step.positions.data_ptr(),
            step.row_seg.data_ptr(), rows, int(window), sc, kw, n_parts, ws.data_ptr(), 0, stream),
            "attention_decode_bf16")
    return True


MASKED_DECODE_BLOCKS = 768    # blocks the decoded rows' key ranges are cut for (3 a compute unit are resident)
MASKED_DECODE_SPLITS = 64     # at most: the adding kernel takes 64 parts


def masked_attention_bf16(q, out, n_heads, n_kv_heads, key_dim, value_dim, cache, page_tokens, block_table, step,
                          mask: str, mask_size: int, sink: bool, scale: float, key_parts: int = 1, sinks=None,
                          gate=None, softcap: float = 0.0, distance_bias=None, keep_first: int = 0,
                          out_scale: float = 1.0) -> bool:
    """Attention with a chunked or sliding mask and an optional sink on the MFMA kernels: segments of several rows on
    the tiled kernel, single rows on the kernel that cuts a row's keys into ranges.  False (nothing done) for sizes
    they do not take; the caller then runs the plain kernel."""
    _ops._gpu(q, out, cache, block_table)
    ldq, ldo = _ops._rows(q, "attention q"), _ops._rows(out, "attention out")
    T = q.shape[0]
    L = _lib.load("tuned")
    f32 = out.dtype == torch.float32
    if gate is not None and gate.dtype != torch.float32:
        return False
    r1, r2 = distance_bias if distance_bias is not None else (None, None)
    r1_p, r2_p = _ops._f32(r1, n_heads, "distance bias r1"), _ops._f32(r2, n_heads, "distance bias r2")
    _ops._check_sinks_gate(sink, sinks, gate, T, n_heads)
    sinks_p = _ops._f32(sinks, n_heads, "sinks")
    gate_p, ldg = (gate.data_ptr(), _ops._rows(gate, "head gate")) if gate is not None else (0, 0)
    if (not scale > 0 or ldq % 8 or ldo % 4 or not _aligned(q, cache) or out.data_ptr() % (16 if f32 else 8)
            or q.dtype != torch.bfloat16 or cache.dtype != torch.bfloat16
            or out.dtype not in (torch.bfloat16, torch.float32)
            or not L.apc_attention_masked_takes(n_heads, n_kv_heads, key_dim, value_dim, page_tokens, key_parts)):
        return False
    _ops._check_key_parts(n_heads, n_kv_heads, key_dim, key_parts)
    _ops._need(q.shape[1] == n_heads * (key_dim // key_parts), "attention: q must be [rows, heads * key_dim / key_parts]")
    _ops._need(out.shape == (T, n_heads * value_dim), "attention out must be [rows, heads * value_dim]")
    _ops._split_pages(cache, n_kv_heads, key_dim, value_dim, page_tokens)
    _ops._need(block_table.dim() == 2 and block_table.dtype == torch.int32 and block_table.is_contiguous(),
               "block table must be contiguous int32 [segments, blocks]")
    _ops._need(step.positions.numel() >= T and step.row_seg.numel() >= T, "step rows differ from q rows")
    code, stream = _ops.MASKS[mask], _ops._stream()
    keep = int(keep_first)
    _ops._need(keep >= 0 and (not keep or mask == "window"), "attention: kept first tokens go with a window")
    if step.n_tiles:
        _lib.check(L.apc_attention_masked_prefill_bf16(
            q.data_ptr(), ldq, out.data_ptr(), ldo, n_heads, n_kv_heads, key_dim, value_dim, cache.data_ptr(),
            page_tokens, block_table.data_ptr(), block_table.shape[1], step.positions.data_ptr(),
            step.row_seg.data_ptr(), step.tile_row0.data_ptr(), step.tile_rows.data_ptr(), step.n_tiles, code,
            int(mask_size), keep, 1 if sink else 0, sinks_p, gate_p, ldg, float(scale), int(key_parts),
            1 if f32 else 0, float(softcap), r1_p, r2_p, float(out_scale), stream), "attention_masked_prefill_bf16")
    if step.n_decode_rows:
        n = step.n_decode_rows
        keys = min(step.max_decode_context, mask_size) if code else step.max_decode_context
        # a row's first pass starts at a multiple of 256 at or below its first key; kept first keys are passes of their own
        passes = -(-(keys + 255) // 256) + -(-min(keep, step.max_decode_context) // 256)
        # (every row sees its keys from 0 on: no such passes, and contexts up to 256 take one launch, 8 us for 17)
        if not code or step.max_decode_context <= mask_size:
            passes = -(-step.max_decode_context // 256)
        splits = max(1, min(passes, MASKED_DECODE_SPLITS, MASKED_DECODE_BLOCKS // max(1, n * n_kv_heads)))
        parts = torch.empty(n * n_heads * splits * (value_dim + 2), dtype=torch.float32, device=q.device)
        _lib.check(L.apc_attention_masked_decode_bf16(
            q.data_ptr(), ldq, out.data_ptr(), ldo, n, n_heads, n_kv_heads, key_dim, value_dim, cache.data_ptr(),
            page_tokens, block_table.data_ptr(), block_table.shape[1], step.positions.data_ptr(),
            step.row_seg.data_ptr(), step.decode_rows.data_ptr() if step.decode_rows is not None else 0, code,
            int(mask_size), keep, 1 if sink else 0, sinks_p, gate_p, ldg, float(scale), splits, parts.data_ptr(),
            int(key_parts), 1 if f32 else 0, float(softcap), r1_p, r2_p, float(out_scale), stream),
            "attention_masked_decode_bf16")
    return True


LINEAR_CHUNK_MIN_ROWS = 5    # segments of at least this many rows make a step run on the kernel of 64-row chunks


def linear_attention_bf16(proj, q_off, k_off, v_off, H, dk, dv, silu, decay, state, step, slots, out,
                          powers=None, rot: int = 0, cos_sin=None, k_scale: float = 1.0) -> bool:
    """Linear attention with a decay on the MFMA kernel that walks a segment in chunks of 64 rows.  False (nothing
    done) for sizes it does not take and for steps whose segments are all short (decoded rows): the caller then runs
    the kernel that walks row by row.  With a rotation or a key scale, q and k of `proj` are first rotated (and k
    scaled) where they lie, in bfloat16: the chunk kernels' operands are 16 bits anyway."""
    ld, ldo = _ops._rows(proj, "projected rows"), _ops._rows(out, "linear attention out")
    L = _lib.load("tuned")
    if (step.max_rows < LINEAR_CHUNK_MIN_ROWS or proj.dtype != torch.bfloat16 or ldo % 4 or not _aligned(proj, out)
            or not L.apc_linear_attention_bf16_takes(ld, q_off, k_off, v_off, H, dk, dv)):
        return False
    if rot or float(k_scale) != 1.0:
        if silu or rot % 16 or (rot and not _aligned(cos_sin)):
            return False
        T = proj.shape[0]
        _lib.check(L.apc_linear_rotate_bf16(proj.data_ptr(), ld, q_off, k_off, H, dk, int(rot),
                                            cos_sin.data_ptr() if rot else 0,
                                            _ops._i32(step.positions, T, "positions") if rot else 0, float(k_scale), T,
                                            _ops._stream()), "linear_rotate_bf16")
    S = step.n_segs
    if powers is None:         # (a caller that keeps the table, as the mixer does, saves this read-back)
        powers = decay_powers(decay.tolist(), proj.device)
    n_chunks, chunks, seg_chunks = _row_chunks(step, proj.device)
    ws = torch.empty((n_chunks, H, dk, dv), dtype=torch.float32, device=proj.device)
    _lib.check(L.apc_linear_attention_bf16(
        proj.data_ptr(), ld, q_off, k_off, v_off, H, dk, dv, 1 if silu else 0,
        _ops._f32(powers, H * (LINEAR_CHUNK_ROWS + 1), "powers of the decay"),
        state.data_ptr(), S, _ops._i32(step.seg_row0, S, "seg_row0"), _ops._i32(step.seg_rows, S, "seg_rows"),
        _ops._i32(slots, S, "slots"), n_chunks, chunks.data_ptr(), seg_chunks.data_ptr(), ws.data_ptr(),
        out.data_ptr(), ldo, _ops._stream()), "linear_attention_bf16")
    return True


SCAN_CHUNK_MIN_ROWS = 5      # as above, for the selective scan


def selective_scan_bf16(x, dt, dt_bias, A, bc, D, z, state, step, slots, out) -> bool:
    """The selective scan over prompt portions, chunks of 64 rows side by side (summaries, a scan over the chunks, the
    outputs).  False (nothing done) for sizes the kernels do not take and for steps whose segments are all short
    (decoded rows): the caller then runs the kernel that walks row by row."""
    L = _lib.load("tuned")
    T, C = out.shape
    N = int(A.shape[1])
    if step.max_rows < SCAN_CHUNK_MIN_ROWS or not L.apc_selective_scan_bf16_takes(C, N):
        return False
    S = step.n_segs
    n_chunks, chunks, seg_chunks = _row_chunks(step, x.device)
    ws = torch.empty((n_chunks, C, N), dtype=torch.float32, device=x.device)
    sums = torch.empty((n_chunks, C), dtype=torch.float32, device=x.device)
    _lib.check(L.apc_selective_scan_bf16(
        x.data_ptr(), _ops._rows(x, "x"), dt.data_ptr(), _ops._rows(dt, "dt"), _ops._f32(dt_bias, C, "dt bias"),
        A.data_ptr(), bc.data_ptr(), _ops._rows(bc, "B and C"), _ops._f32(D, C, "D"), z.data_ptr(), _ops._rows(z, "z"),
        state.data_ptr(), C, N, S, _ops._i32(step.seg_row0, S, "seg_row0"), _ops._i32(step.seg_rows, S, "seg_rows"),
        _ops._i32(slots, S, "slots"), n_chunks, chunks.data_ptr(), seg_chunks.data_ptr(), ws.data_ptr(),
        sums.data_ptr(), out.data_ptr(), _ops._rows(out, "out"), _ops._stream()), "selective_scan_bf16")
    return True


DELTA_CHUNK_MIN_ROWS = 5     # as above, for the gated delta rule and the gated recurrence


def delta_rule_bf16(rows, ld, q_off, k_off, v_off, H, G, dk, dv, ba, ldba, a_off, b_off, A, dt_bias, state, step, slots,
                    out, ldo) -> bool:
    """The gated delta rule over prompt portions in chunks of 64 rows on MFMA: every chunk's factors side by side, then a
    walk over the chunks.  False (nothing done) for sizes the kernels do not take and for steps whose segments are all
    short (decoded rows): the caller then runs the kernel that walks row by row."""
    L = _lib.load("tuned")
    if (step.max_rows < DELTA_CHUNK_MIN_ROWS or not _aligned(rows)
            or not L.apc_delta_rule_bf16_takes(ld, q_off, k_off, H, G, dk, dv)):
        return False
    S = step.n_segs
    n_chunks, chunks, seg_chunks = _row_chunks(step, rows.device)
    fact = torch.empty(n_chunks * L.apc_delta_rule_fact_size(H), dtype=torch.bfloat16, device=rows.device)
    coef = torch.empty(n_chunks * L.apc_delta_rule_coef_size(H), dtype=torch.float32, device=rows.device)
    kt = torch.empty(n_chunks * G * dk * LINEAR_CHUNK_ROWS, dtype=torch.bfloat16, device=rows.device)
    _lib.check(L.apc_delta_rule_bf16(
        rows.data_ptr(), ld, q_off, k_off, v_off, H, G, dk, dv, ba.data_ptr(), ldba, a_off, b_off, _ops._f32(A, H, "A"),
        _ops._f32(dt_bias, H, "dt bias"), float(dk) ** -0.5, state.data_ptr(), S, _ops._i32(step.seg_row0, S, "seg_row0"),
        _ops._i32(step.seg_rows, S, "seg_rows"), _ops._i32(slots, S, "slots"), n_chunks, chunks.data_ptr(),
        seg_chunks.data_ptr(), fact.data_ptr(), coef.data_ptr(), kt.data_ptr(), out.data_ptr(), ldo, _ops._stream()),
        "delta_rule_bf16")
    return True


def gated_recurrence_bf16(u, z, z_bias, blocks: int, rate, y, y_bias, state, step, slots, out, out_scale: float) -> bool:
    """The gated linear recurrence over prompt portions, chunks of 64 rows side by side (summaries, a scan over the
    chunks, the outputs).  False (nothing done) as above."""
    L = _lib.load("tuned")
    T, C = out.shape
    ldu, ldz, ldy, ldo = _ops._rows(u, "u"), _ops._rows(z, "gate logits"), _ops._rows(y, "y"), _ops._rows(out, "out")
    if (step.max_rows < DELTA_CHUNK_MIN_ROWS or not L.apc_gated_recurrence_bf16_takes(C, blocks, ldu, ldz, ldy, ldo)
            or any(t.data_ptr() % 4 for t in (u, y, out)) or z.data_ptr() % 8):
        return False
    S = step.n_segs
    n_chunks, chunks, seg_chunks = _row_chunks(step, u.device)
    ws = torch.empty((10, n_chunks, C), dtype=torch.float32, device=u.device)
    _lib.check(L.apc_gated_recurrence_bf16(
        u.data_ptr(), ldu, z.data_ptr(), ldz, _ops._f32(z_bias, 2 * C, "gate biases"), blocks, _ops._f32(rate, C, "rate"),
        y.data_ptr(), ldy, _ops._f32(y_bias, C, "y bias"), float(out_scale), state.data_ptr(), C, S,
        _ops._i32(step.seg_row0, S, "seg_row0"), _ops._i32(step.seg_rows, S, "seg_rows"), _ops._i32(slots, S, "slots"),
        n_chunks, chunks.data_ptr(), seg_chunks.data_ptr(), ws.data_ptr(), out.data_ptr(), ldo,
        _ops._stream()), "gated_recurrence_bf16")
    return True


def recurrent_step_bf16(x, y, in_bias, conv_w, conv_b, conv_state, conv_slots, w_gates, z_bias, blocks: int, rate, y_bias, state, slots,
                        step, out, out_scale: float) -> bool:
    """One row of every request through the convolution, the gates' products and the recurrence in one launch; False
    (nothing done) for sizes that it does not take."""
    L = _lib.load("tuned")
    T, C = out.shape
    taps = int(conv_w.shape[1])
    ldx, ldy, ldo = _ops._rows(x, "conv input"), _ops._rows(y, "y"), _ops._rows(out, "out")
    S = step.n_segs
    if (conv_state is None or conv_slots is None or S != T or not L.apc_recurrent_step_bf16_takes(T, C, blocks, taps, ldx, ldy, ldo)
            or not _aligned(x, conv_state, state, z_bias, rate, w_gates.data) or (y_bias is not None and not _aligned(y_bias))
            or any(t.data_ptr() % 8 for t in (y, out))):
        return False
    w = C // blocks
    _ops._gpu(x, y, conv_w, conv_state, w_gates.data, state, out)
    _ops._need(x.shape[0] == T and x.shape[1] >= C and y.shape == (T, C), "recurrent step: x and y hold the channels of every row")
    _ops._need(w_gates.H == blocks and w_gates.N == 2 * w and w_gates.K == w, "recurrent step: a matrix [2 w, w] for every part")
    _ops._need(conv_w.shape[0] == C and conv_w.dtype == torch.float32 and conv_w.is_contiguous(), "recurrent step: float32 [channels, taps]")
    _ops._need(conv_state.dtype == torch.float32 and conv_state.is_contiguous() and tuple(conv_state.shape[1:]) == (taps - 1, C)
               and state.dtype == torch.float32 and state.is_contiguous() and tuple(state.shape[1:]) == (C,),
               "recurrent step: states must be float32 [slots, taps - 1, channels] and [slots, channels]")
    _lib.check(L.apc_recurrent_step_bf16(
        x.data_ptr(), ldx, y.data_ptr(), ldy, _ops._f32(in_bias, C, "input bias"), conv_w.data_ptr(), _ops._f32(conv_b, C, "bias"), taps,
        conv_state.data_ptr(), w_gates.data.data_ptr(), _ops._f32(z_bias, 2 * C, "gate biases"), blocks, _ops._f32(rate, C, "rate"),
        _ops._f32(y_bias, C, "y bias"), out_scale, state.data_ptr(), T, C, _ops._i32(step.row_seg, T, "row_seg"),
        _ops._i32(conv_slots, S, "slots"), _ops._i32(slots, S, "slots"), out.data_ptr(), ldo, _ops._stream()), "recurrent_step_bf16")
    return True


LINEAR_CHUNK_ROWS = 64


def decay_powers(decay, device) -> torch.Tensor:
    """float32 [heads, 65]: decay^0 .. decay^64 of every head (`decay`: the heads' numbers), formed in double precision
    on the host and rounded once: what the chunk kernels multiply scores, outputs and states with."""
    rows = [[float(d) ** n for n in range(LINEAR_CHUNK_ROWS + 1)] for d in decay]
    return torch.tensor(rows, dtype=torch.float64).to(torch.float32).to(device).contiguous()


def _row_chunks(step, device):
    """(chunks in all, int32 [chunks][2] (segment, first row in it), int32 [segments][2] (a segment's first chunk, its
    chunks)) of a step's segments cut into chunks of 64 rows: made on the host from the step's own lists, once a step
    (every layer of the step asks for the same)."""
    made = getattr(step, "_row_chunks", None)
    if made is None:
        import numpy as np
        chunks, per_seg = [], []
        for s, n in enumerate(step.host_rows):
            per_seg.append((len(chunks), -(-n // LINEAR_CHUNK_ROWS)))
            chunks += [(s, c0) for c0 in range(0, n, LINEAR_CHUNK_ROWS)]
        flat = np.asarray(chunks + per_seg, dtype=np.int32).reshape(-1)
        dev = torch.from_numpy(flat).to(device)
        made = (len(chunks), dev[:2 * len(chunks)], dev[2 * len(chunks):])
        step._row_chunks = made
    return made


class PackedExperts:
    """The matrices of a layer's experts in the tiled layout of the MFMA kernels: `data` holds, for every expert, the
    tiles of its matrices (`per_expert` of them: gate and up, or down alone), each packed like a `PackedWeight`."""

    def __init__(self, data: torch.Tensor, n_experts: int, N: int, K: int, per_expert: int = 1):
        self.data, self.E, self.N, self.K, self.per_expert = data, n_experts, N, K, per_expert


# pairs an expert on average from which a row tile holds 64 and 128 rows instead of 16 (and the products run on the
# tiled kernel through LDS instead of streaming an expert's matrices once a tile)
ROUTED_TILE_64_MIN, ROUTED_TILE_128_MIN = 24, 96


def pack_experts(gate_up: torch.Tensor, down: torch.Tensor):
    """[E, 2 F, D] (gate rows, then up rows; [E, F, D] for experts without a gate) and [E, D, F] bfloat16 ->
    (PackedExperts, PackedExperts), or None for sizes the kernels do not take."""
    from .packing import pack_mfma
    E, D, F = down.shape
    gated = gate_up.shape[1] == 2 * F
    if not _lib.load("tuned").apc_routed_bf16_takes(E, F, D):
        return None
    firsts = (slice(0, F), slice(F, 2 * F)) if gated else (slice(0, F),)
    gu = torch.stack([torch.stack([pack_mfma(gate_up[e, s].contiguous()).data for s in firsts])
                      for e in range(E)]).contiguous()
    dn = torch.stack([pack_mfma(down[e].contiguous()).data for e in range(E)]).contiguous()
    return PackedExperts(gu, E, F, D, len(firsts)), PackedExperts(dn, E, D, F)


def routed_experts_bf16(h, w_gate_up: PackedExperts, w_down: PackedExperts, E: int, F: int, ids, weights, K: int,
                        y, kind: int = 0, alpha: float = 1.0, limit: float = 0.0, weight_input: bool = False) -> None:
    """The chosen experts of every row on the MFMA kernels (pairs sorted by expert on the GPU, nothing read back).
    `weight_input`: a pair's weight multiplies the expert's input instead of its output."""
    T, D = h.shape
    _ops._gpu(h, w_gate_up.data, w_down.data, ids, weights, y)
    _ops._need(h.dtype == torch.bfloat16 and (w_gate_up.E, w_gate_up.N, w_gate_up.K) == (E, F, D)
               and (w_down.E, w_down.N, w_down.K) == (E, D, F) and w_gate_up.per_expert == (1 if kind == 2 else 2), "routed experts: matrices do not fit the sizes")
    L = _lib.load("tuned")
    n_pairs = T * K
    tile_rows = 128 if n_pairs >= ROUTED_TILE_128_MIN * E else 64 if n_pairs >= ROUTED_TILE_64_MIN * E else 16
    max_tiles = L.apc_routed_max_tiles(n_pairs, E, tile_rows)
    dev = h.device
    work = torch.empty(2 * n_pairs + 3 * max_tiles + 1, dtype=torch.int32, device=dev)
    act = torch.empty((n_pairs, F), dtype=torch.bfloat16, device=dev)
    ys = torch.empty((n_pairs, D), dtype=torch.float32, device=dev)
    hs = torch.empty((n_pairs, D), dtype=torch.bfloat16, device=dev) if tile_rows != 16 else None
    _lib.check(L.apc_routed_experts_bf16(
        h.data_ptr(), _ops._rows(h, "h"), w_gate_up.data.data_ptr(), w_down.data.data_ptr(), E, F, D,
        _ops._i32(ids, n_pairs, "ids"), _ops._f32(weights, n_pairs, "weights"), K, T, tile_rows, work.data_ptr(),
        act.data_ptr(), ys.data_ptr(), hs.data_ptr() if hs is not None else 0, y.data_ptr(), _ops._rows(y, "y"),
        int(kind), float(alpha), float(limit), 1 if weight_input else 0, _ops._stream()),
        "routed_experts_bf16")


def rotary_pages_bf16(q, ldq, q_off, H, dq, q_rot0, q_out, ldqo, ka, ldka, ka_off, da, kb, ldkb, kb_off, db, kb_shared,
                      k_rot0, v, ldv, v_off, dv, G, rot, cos_sin, step, block_table, cache, page_tokens, q_norm_w=None,
                      k_norm_w=None, norm_eps: float = 0.0) -> bool:
    """Heads put together, rotated and written into the pages on 16-byte accesses (bfloat16 rows and pages; the second
    key part may be float32 rows); False (nothing done) for sizes the kernel does not take."""
    L = _lib.load("tuned")
    T = q.shape[0]
    if H <= 0 or G <= 0 or (kb is not None and kb.dtype not in (torch.bfloat16, torch.float32)):
        return False
    if not L.apc_rotary_pages_bf16_takes(ldq, q_off, dq, q_rot0, ldqo, ldka, ka_off, da, ldkb, kb_off, db, k_rot0, ldv,
                                         v_off, dv, rot):
        return False
    if not _aligned(q, q_out, ka, v, cache) or (kb is not None and not _aligned(kb)) or (rot and not _aligned(cos_sin)):
        return False
    if q_norm_w is not None or k_norm_w is not None:
        # a wave a head: no second key part, heads of up to 512 elements
        if kb is not None or db or max(dq, da, dv) > 512 or not all(w is None or _aligned(w) for w in (q_norm_w, k_norm_w)):
            return False
    _lib.check(L.apc_rotary_pages_bf16(
        q.data_ptr(), ldq, q_off, H, dq, q_rot0, q_out.data_ptr(), ldqo, ka.data_ptr(), ldka, ka_off, da,
        kb.data_ptr() if kb is not None else 0, 1 if kb is not None and kb.dtype == torch.float32 else 0, ldkb, kb_off,
        db, 1 if kb_shared else 0, k_rot0, v.data_ptr(), ldv, v_off, dv, G, rot, cos_sin.data_ptr() if rot else 0,
        _ops._i32(step.positions, T, "positions"), _ops._i32(step.row_seg, T, "row_seg"), block_table.data_ptr(),
        block_table.shape[1], cache.data_ptr(), page_tokens, T, _ops._f32(q_norm_w, dq, "q norm weight"),
        _ops._f32(k_norm_w, da + db, "k norm weight"), float(norm_eps), _ops._stream()), "rotary_pages_bf16")
    return True


# --------------------------------------------------------------------------- a matrix of its own for every head
class PackedHeads:
    """[heads, N, K] matrices in the tiled layout: `data` [heads, bands, chunks, 64, 8]."""

    def __init__(self, data: torch.Tensor, H: int, N: int, K: int):
        self.data, self.H, self.N, self.K = data, H, N, K


def pack_heads(w: torch.Tensor, a_head: int, out_head: int):
    """[H, N, K] bfloat16 -> PackedHeads, or None where the kernel does not take the heads' places in the rows (`a_head`
    elements apart in the product's input, `out_head` in its output)."""
    from .packing import can_pack, pack_mfma
    if not can_pack(w[0]) or a_head % 8 or out_head % 4:
        return None
    H, N, K = w.shape
    return PackedHeads(torch.stack([pack_mfma(w[h].contiguous()).data for h in range(H)]).contiguous(), H, N, K)


def heads_linear_bf16(a: torch.Tensor, a_head: int, w: PackedHeads, out: torch.Tensor, out_head: int, gate=None) -> None:
    _ops._gpu(a, w.data, out)
    lda, ldo = _ops._rows(a, "heads_linear a"), _ops._rows(out, "heads_linear out")
    T = a.shape[0]
    f32 = out.dtype == torch.float32
    _ops._need(a.dtype == torch.bfloat16 and (f32 or out.dtype == torch.bfloat16) and out.shape[0] == T
               and (w.H - 1) * a_head + w.K <= a.shape[1] and (w.H - 1) * out_head + w.N <= out.shape[1],
               "heads_linear: bfloat16 rows that hold the heads' ranges")
    ldg = _ops._rows(gate, "gate") if gate is not None else 0
    _ops._need(gate is None or (gate.dtype == torch.bfloat16 and ldg % 4 == 0 and gate.data_ptr() % 8 == 0),
               "heads_linear_bf16: the gate's logits are bfloat16 rows of a stride that is a multiple of 4")
    _ops._need(lda % 8 == 0 and ldo % 4 == 0 and _aligned(a) and out.data_ptr() % (16 if f32 else 8) == 0,
               "heads_linear_bf16: rows of a stride that is a multiple of 8 (out: 4), aligned")
    L = _lib.load("tuned")
    _lib.check(L.apc_heads_gemm_bf16(a.data_ptr(), lda, int(a_head), w.data.data_ptr(), out.data_ptr(), ldo, int(out_head),
                                     1 if f32 else 0, gate.data_ptr() if gate is not None else 0, ldg, T, w.H, w.N, w.K,
                                     _ops._stream()), "heads_gemm_bf16")


def latent_rows_bf16(proj, ld, H, dn, dr, kv, ldkv, c_off, R, norm_w, eps, cos_sin, step, block_table, pages,
                     page_tokens, q_out, ldq) -> bool:
    """The same on 16-byte accesses; False (nothing done) for sizes the kernel does not take."""
    L = _lib.load("tuned")
    T = proj.shape[0]
    if not L.apc_latent_rows_bf16_takes(ld, dn, dr, ldkv, c_off, R, ldq) or not _aligned(proj, kv, pages, q_out, cos_sin):
        return False
    _lib.check(L.apc_latent_rows_bf16(
        proj.data_ptr(), ld, H, dn, dr, kv.data_ptr(), ldkv, c_off, R, _ops._f32(norm_w, R, "norm weight"), float(eps), cos_sin.data_ptr(),
        _ops._i32(step.positions, T, "positions"), _ops._i32(step.row_seg, T, "row_seg"), block_table.data_ptr(),
        block_table.shape[1], pages.data_ptr(), page_tokens, q_out.data_ptr(), ldq, T, _ops._stream()), "latent_rows_bf16")
    return True


LATENT_BLOCKS = 256          # blocks that the keys of few rows are cut for (a block a compute unit at a latent of 512)
LATENT_SPLITS_MAX = 128      # (the adding kernel takes up to 256; 128 was the fastest for one row over 32,768 keys)
LATENT_DECODE_TILES = 2      # key tiles that a range of a decoded row's keys must keep
LATENT_RANGE_TILES = 8       # key tiles (of 64) that a range of a prompt tile's keys must keep


def latent_attention_bf16(q, out, n_heads: int, rank: int, rot_dim: int, pages, page_tokens: int, block_table, step,
                          scale: float) -> bool:
    """Attention of all heads over cached latents on MFMA: tiles of prompt rows, then single rows.  False (nothing done)
    for sizes the kernel does not take."""
    _ops._gpu(q, out, pages, block_table)
    T, H, R, dr = q.shape[0], int(n_heads), int(rank), int(rot_dim)
    L = _lib.load("tuned")
    if (q.dtype != torch.bfloat16 or pages.dtype != torch.bfloat16 or out.dtype != torch.bfloat16
            or not q.is_contiguous() or not out.is_contiguous() or not _aligned(q, out, pages)
            or not L.apc_latent_attention_takes(H, R, dr, page_tokens)):
        return False
    _ops._need(tuple(q.shape) == (T, H * (R + dr)) and tuple(out.shape) == (T, H * R), "latent attention: q [rows, heads * "
               "(rank + rot_dim)], out [rows, heads * rank]")
    _ops._latent_pages(pages, R + dr, page_tokens, block_table)
    _ops._need(step.positions.numel() >= T and step.row_seg.numel() >= T, "step rows differ from q rows")

    def run(row0, rows, n: int, max_rows: int, splits: int, what: str) -> None:
        parts = ml = None
        if splits > 1:
            parts = torch.empty((T * H, splits, R), dtype=torch.float32, device=q.device)
            ml = torch.empty((T * H, splits, 2), dtype=torch.float32, device=q.device)
        _lib.check(L.apc_latent_attention_bf16(
            q.data_ptr(), out.data_ptr(), H, R, dr, pages.data_ptr(), page_tokens, block_table.data_ptr(),
            block_table.shape[1], step.positions.data_ptr(), step.row_seg.data_ptr(),
            row0.data_ptr() if row0 is not None else 0, rows.data_ptr() if rows is not None else 0, n, max_rows, splits,
            parts.data_ptr() if parts is not None else 0, ml.data_ptr() if ml is not None else 0, float(scale),
            _ops._stream()), what)

    if step.n_tiles:
        most = min(step.max_rows, _ops.attention_tile_rows(torch.bfloat16))
        blocks = step.n_tiles * -(-most * H // 64)
        keys = max([p + n for p, n in zip(step.host_pos0, step.host_rows) if n > 1] or [step.max_context])
        splits = max(1, min(LATENT_BLOCKS // blocks, -(-keys // 64) // LATENT_RANGE_TILES, LATENT_SPLITS_MAX))
        run(step.tile_row0, step.tile_rows, step.n_tiles, most, splits, "latent_attention_bf16 (prompt rows)")
    if step.n_decode_rows:
        n = step.n_decode_rows
        blocks = n * -(-H // (64 if H > 32 else 32))
        splits = max(1, min(LATENT_BLOCKS // blocks, -(-step.max_decode_context // (64 * LATENT_DECODE_TILES)), LATENT_SPLITS_MAX))
        run(step.decode_rows, None, n, 1, splits, "latent_attention_bf16 (decoded rows)")
    return True
