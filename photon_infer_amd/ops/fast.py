"""Dispatch to the bfloat16 matrix-core kernels (module "bf16").

Each function returns True when it ran the operation and False when the sizes are not
ones its kernels take, in which case the caller uses the general kernel.

Which kernel takes what:
  * matrix products: K and the row strides multiples of 8, 16-byte aligned operands;
    up to 128 rows go to the weight-streaming kernels (k split over blocks where the output
    is narrow), more rows to the tile kernels;
  * attention: pages of a multiple of 16 tokens; a batch of single tokens with at most 16 heads
    per kv head goes to the key-split decode kernel (head_dim a multiple of 16 up to 256; for
    64 and 128 straight from the q|k|v projection), any other batch to the tile kernel
    (head_dim a multiple of 16 up to 256), its single tokens to the decode kernel.
"""
from __future__ import annotations

import ctypes
import functools
from dataclasses import dataclass
from typing import Any, Callable, Dict, List, Optional, Sequence, Tuple

import numpy as np
import torch

from ..errors import KernelError
from . import _lib
from .workspace import GEMM_PART_FLOATS, KernelWorkspace, KeyRanges, LeftNorm, Partials, PendingUpdate

EPI_BF16, EPI_F32, EPI_ACCUM, EPI_SWIGLU = 0, 1, 2, 3
SKINNY_MAX_ROWS = 128          # up to this many tokens the weight-streaming kernels serve a product (measured against the tile kernel)
ROWS_PER_BLOCK = 32            # weight rows per block of the skinny kernel
BLOCKS_PER_UNIT = 2            # blocks of it wanted per compute unit to keep HBM busy (measured: 512 on 256 units; 384 and 768 are slower)
SHARED_FROM_TOKENS = 32        # more tokens than this: the skinny kernel that shares activations per block (from 17 on for large matrices: pi_gemm_skinny_shares) ...
SHARED_ROWS_PER_BLOCK = 64     # ... with this many weight rows per block, and no more blocks than compute units (100 tokens, 3,072 x 8,192:
                               # 22.8 us in six pieces on 288 blocks, 16.9 in five on 240; 6,144 x 4,096 22.8 in three, 18.7 in two), though
                               # a unit would hold two: 64 tokens, k 4,096, blocks for half the units or more in one piece and in two, 8,256
                               # rows 29.7 and 32.0, 9,216 29.2 and 31.3, 12,160 29.4 and 31.1, 14,720 33.2 and 35.4; the same at 100 tokens
                               # (35.7 and 39.0, 35.4 and 38.0, 35.4 and 37.6, 39.1 and 41.7), and at k of 2,048 and 8,192
FEW_TOKENS = 16                # up to this many tokens a product whose weights have a streaming copy may take all of k in a block (pi_gemm_rows)
FEW_TOKENS_WHOLE_K = 4096      # ... and does in the place of pieces that a kernel of its own would add, up to this k (M = 1 / 12: 1,024 x 2,048 5.4 / 5.9
                               # us in pieces and 3.3 / 4.2, 4,384 x 2,048 8.8 / 9.5 and 6.3 / 7.4, 6,560 x 3,072 12.7 / 13.7 and 9.6 / 10.6; 2,048 x
                               # 8,192 11 / 11 and 10 / 13)
RING_MAX_STRIDE = 1 << 21      # elements between rows up to which that kernel's byte offsets fit 31 bits
FLOAT32_ROWS = 32              # up to this many rows a float32 product goes to the weight-streaming kernel
FLOAT32_MAX_STRIDE = 1 << 21   # floats between rows up to which the float32 kernels' offsets inside a tile fit 32 bits
DEFAULT_UNITS = 256            # compute units assumed where no device can be asked (an MI355X)
PIECES_WORTH = 0.95            # q, k, v of a prompt portion are left in k pieces too where that takes no more than this share of the time:
                               # their reader, the rotation, then reads float32 pieces instead of one bfloat16 tensor
TILE_HEAD_DIMS = tuple(range(16, 257, 16))         # head sizes of the prompt-attention tile kernel (above 128: rounds of 64 keys, 16 columns per wave)
DECODE_HEAD_DIMS = tuple(range(16, 257, 16))       # head sizes of the key-split decode kernel
FUSED_DECODE_HEAD_DIMS = (64, 128)                 # ... and of its form that starts from the q|k|v projection (whole halves of a head per fragment)
MAX_DECODE_SPLITS = 64         # the combine kernel holds one key range per lane
DECODE_WAVES_PER_UNIT = 2      # waves of the decode attention kernel per compute unit that fill the chip (measured at batch 1 to 64: more is never faster)
DECODE_MIN_KEYS_PER_SPLIT = 128
RANGES_TO_SHARE = 32           # ranges of all requests from which on two waves of a block share one (decode_range_waves) ...
RANGES_SHARED_UP_TO = 4        # ... in steps of up to so many requests
# Waves that share a block's keys, against ranges with their merging kernel or one wave (lists of attention times, 32 heads, 8 kv
# heads, 600 to 4,096 keys each).  Blocks have to fill their rounds over the units this far: 384 of them, 1.5 rounds, at 4,096
# keys 75.7 -> 81.0 us (up to 1,024 keys 23.8 -> 21.4), 320 at head size 128 126 -> 140; 192, three quarters of one round,
# 38.6 -> 33.7.  Without ranges to replace only at two rounds (three, head size 128: 278 -> 296 at 4,096 keys, 42 -> 46 at 600),
# from contexts on that are longer than so many keys per 64 features (64 requests of 600 at head size 128 29.8 -> 30.2), and
# for lengths that are uneven: 64 requests of 2,000 to 4,000 keys 83 -> 76, of 4,096 each 96.5 -> 99.5 and with the second
# waves gone at once 97.  From 10 % between the longest and the mean on the waves gain.
DECODE_WAVES_FILL, DECODE_WAVES_FILL_LONG, DECODE_WAVES_LONG, DECODE_WAVES_MIN_KEYS = 0.75, 0.8, 1024, 512
PLAIN_HEADS = (None, None, None, 0, 0.0, 1.0, 0, 0)   # a decode attention's options: none
UNEVEN = 1.1                   # longest context over the mean from which a step's lengths are uneven


def _stream() -> int:
    return _lib.current_stream()


@functools.lru_cache(maxsize=None)
def _units_of(index: int) -> int:
    return int(torch.cuda.get_device_properties(index).multi_processor_count)


def compute_units() -> int:
    """Compute units of the current device: the split rules below count blocks and waves in
    multiples of it (256 on an MI355X, where they were measured)."""
    try:
        return _units_of(_lib.current_device())
    except Exception:                    # no device in this process (rules asked for on the host)
        return DEFAULT_UNITS


def _gemm_ok(a, w, K, lda, ldw) -> bool:
    return (K % 8 == 0 and lda % 8 == 0 and ldw % 8 == 0 and a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and not (SHARED_FROM_TOKENS < a.shape[0] <= SKINNY_MAX_ROWS and max(lda, ldw) >= RING_MAX_STRIDE))


def _skinny_splits(M: int, N: int, K: int) -> int:
    return _skinny_splits_of(M, N, K, compute_units())


def _far_rows_splits(M: int, N: int, K: int) -> int:
    """The same where rows are too far apart for the kernel that shares activations."""
    return _skinny_splits_of(M, N, K, compute_units(), RING_MAX_STRIDE)


@functools.lru_cache(maxsize=4096)
def _skinny_splits_of(M: int, N: int, K: int, units: int, stride: int = 0) -> int:
    if _lib.load("bf16").pi_gemm_skinny_shares(M, N, K, stride, stride):
        # the kernel that shares an activation tile per block: at most one block per compute unit
        splits = units // -(-N // SHARED_ROWS_PER_BLOCK)
    else:
        splits = -(-BLOCKS_PER_UNIT * units // -(-N // ROWS_PER_BLOCK))
    splits = max(1, min(splits, K // 256))
    while splits > 1 and splits * M * N > GEMM_PART_FLOATS:
        splits -= 1
    return splits


@functools.lru_cache(maxsize=4096)
def _tile_shape_of(M: int, N: int, K: int, splits: int, units: int) -> int:
    return _lib.load("bf16").pi_gemm_mfma_shape(M, N, K, splits, units)


@functools.lru_cache(maxsize=4096)
def _tile_splits_of(M: int, N: int, K: int, units: int, worth: float, norm: bool = True) -> int:
    return _lib.load("bf16").pi_gemm_mfma_splits(M, N, K, units, GEMM_PART_FLOATS, worth, norm)


def _tile_shape(M: int, N: int, K: int, splits: int) -> int:
    """The block tile (its code, csrc/tile_plan.h) that takes the least time for the product in ``splits`` pieces."""
    return _tile_shape_of(M, N, K, splits, compute_units())


def _tile_splits(M: int, N: int, K: int) -> int:
    """k-split of the tile kernels for a product whose reader, a norm, adds the pieces: as many as take the least time
    together with the pieces' way through memory."""
    return _tile_splits_of(M, N, K, compute_units(), 1.0)


def flush(ws: Optional[KernelWorkspace]) -> None:
    """The product scratch is about to be reused: apply the update that still lives in it."""
    if ws is None or ws.pending is None:
        return
    p, ws.pending = ws.pending, None
    reduce_into(p.target, p.pieces, accumulate=p.accumulate)
    ws.counts_of(p.pieces)["flushed"] += 1


def _piece_buffer(ws: Optional[KernelWorkspace], floats: int, device) -> torch.Tensor:
    """Where the pieces of a split product go: the workspace's buffer (whose last tenant is
    applied first), or memory of this call's own."""
    if ws is None:
        return torch.empty(floats, dtype=torch.float32, device=device)
    if floats > GEMM_PART_FLOATS:
        # the split rules never ask for more; a kernel writing pieces past the buffer would fault the GPU
        raise KernelError(f"pieces of a split product need {floats} floats, the workspace holds {GEMM_PART_FLOATS}")
    flush(ws)
    return ws.gemm_part


def _streamed(ws: Optional[KernelWorkspace], w, N: int, K: int, ldw: int):
    """(address, tiled) of the weight matrix for the weight-streaming kernels: its copy in their
    own order when the workspace keeps one, else the matrix itself."""
    if ws is not None and ws.stream_copies and ldw == K:
        copy = ws.stream_copy_of(w, N, K)
        if copy is not None:
            return copy.data_ptr(), 1
    return w.data_ptr(), 0


def applies_root(left: LeftNorm, w, ws: Optional[KernelWorkspace]) -> bool:
    """Whether a product of the norm that ``left`` stands for with ``w`` [N, K] is one that applies the root itself: ``_rows``
    does, which reads the streaming copy.  For any other the norm is made whole, and the product takes its ordinary way."""
    M, K = left.shape
    return (ws is not None and w.dim() == 2 and w.dtype == torch.bfloat16 and M <= FEW_TOKENS and w.shape[1] == K and K < RING_MAX_STRIDE
            and w.is_contiguous() and left.h.is_contiguous() and _gemm_ok(left.h, w, K, K, K) and ws.has_stream_copy(w))


def _rows(out_ptr: int, epilogue: int, ldc: int, a, w, M, N, K, lda, ldw, ws: Optional[KernelWorkspace], left: Optional[LeftNorm] = None) -> bool:
    """A product of up to 16 tokens by the kernel whose blocks take all of k, which reads the weights' streaming copy: False, and
    nothing done, without one.  ``left``: what ``a`` is the ``h`` of."""
    w_ptr, tiled = _streamed(ws, w, N, K, ldw)
    if not tiled or max(lda, K) >= RING_MAX_STRIDE:
        return False
    _lib.call("bf16", "pi_gemm_rows", out_ptr, epilogue, ldc, a.data_ptr(), lda, w_ptr, M, N, K, None if left is None else left.sums.data_ptr(),
              0 if left is None else left.count, 0.0 if left is None else left.eps, _stream())
    if left is not None:
        ws.counts["left_norms_read"] += 1
    return True


def _skinny(out_ptr: int, epilogue: int, ldc: int, a, w, M, N, K, lda, ldw, splits: int,
            ws: Optional[KernelWorkspace], pieces_ws: bool = True) -> Optional[Partials]:
    """Run the weight-streaming kernel; returns the pieces when the product was split.
    ``pieces_ws`` False: the workspace is only asked for the weights' streaming copy."""
    if splits == 1 and M <= FEW_TOKENS and _rows(out_ptr, epilogue, ldc, a, w, M, N, K, lda, ldw, ws):
        return None
    buf = _piece_buffer(ws if pieces_ws else None, splits * M * N, a.device) if splits > 1 else None
    made = ctypes.c_int(0)
    w_ptr, tiled = _streamed(ws, w, N, K, ldw)
    _lib.call("bf16", "pi_gemm_skinny", out_ptr, epilogue, ldc, a.data_ptr(), lda, w_ptr, ldw, M, N, K, splits,
              None if buf is None else buf.data_ptr(), 0 if buf is None else buf.numel(), ctypes.addressof(made), tiled, _stream())
    if made.value > 1:
        if ws is not None:
            ws.counts["split_products"] += 1
        return Partials(buf, made.value, M, N)
    return None


def _tiles_in_pieces(a, w, M, N, K, lda, ldw, splits: int, ws: Optional[KernelWorkspace]) -> Optional[Partials]:
    """The tile kernel with its k-range split: float32 pieces, nothing else written."""
    buf = _piece_buffer(ws, splits * M * N, a.device)
    made = _lib.load("bf16").pi_gemm_mfma_pieces(K, splits)
    _lib.call("bf16", "pi_gemm_mfma", buf.data_ptr(), EPI_F32, N, a.data_ptr(), lda, w.data_ptr(), ldw, M, N, K, splits,
              _tile_shape(M, N, K, splits), _stream())
    if ws is not None:
        ws.counts["split_products"] += 1
    return Partials(buf, made, M, N)


def reduce_into(out: torch.Tensor, p: Partials, accumulate: bool) -> None:
    epilogue = EPI_ACCUM if accumulate else (EPI_BF16 if out.dtype == torch.bfloat16 else EPI_F32)
    _lib.call("core", "pi_splitk_reduce", out.data_ptr(), epilogue, out.stride(0), p.part.data_ptr(), p.splits, p.M, p.N,
              _stream())


@functools.lru_cache(maxsize=4096)
def _finish_blocks(M: int, N: int, K: int) -> int:
    return _lib.load("bf16").pi_gemm_finish_blocks(M, N, K)


@functools.lru_cache(maxsize=4096)
def _finish_ranges_blocks(M: int, N: int, heads: int, head_dim: int, count: int) -> int:
    return _lib.load("bf16").pi_gemm_finish_ranges_blocks(M, N, heads, head_dim, count)


def _finish(out, a, w, M, N, K, lda, ldw, next_norm, ws: KernelWorkspace, bias=None) -> bool:
    """out += a @ w^T of a few tokens by the kernel that also makes the next norm but for its root, left in the workspace (in
    the place of pieces of k, whose order of sums hangs on the step anyway; a product that is not cut keeps the one order that
    steps up to 16 tokens have, and up to 32 on matrices below 20 million elements); False, and nothing done, where it does not
    take the product or the weights have no streaming copy.  ``a`` may be ``KeyRanges``, where the kernel merges as many.  ``bias`` (float32 [N], not with ranges): added besides."""
    weight, eps = next_norm
    ranges = a if isinstance(a, KeyRanges) else None
    blocks = _finish_blocks(M, N, K) if ranges is None else _finish_ranges_blocks(M, N, ranges.heads, ranges.head_dim, ranges.count)
    if not blocks or out.dtype != torch.float32 or not weight.is_contiguous() or weight.numel() != N or lda >= RING_MAX_STRIDE:
        return False
    w_ptr, tiled = _streamed(ws, w, N, K, ldw)
    if not tiled:
        return False
    h = torch.empty((M, N), dtype=torch.bfloat16, device=out.device)
    sums = torch.empty((M, blocks), dtype=torch.float32, device=out.device)
    norm = (weight.data_ptr(), 0 if weight.dtype == torch.float32 else 1, h.data_ptr(), sums.data_ptr(), sums.numel())
    if ranges is None:
        _lib.call("bf16", "pi_gemm_finish", out.data_ptr(), a.data_ptr(), lda, w_ptr, *norm, None if bias is None else bias.data_ptr(), M, N, K, _stream())
    else:
        _lib.call("bf16", "pi_gemm_finish_ranges", out.data_ptr(), ranges.part.data_ptr(), ranges.heads, ranges.head_dim, ranges.count, w_ptr, *norm,
                  M, N, _stream())
        ws.counts["ranges_merged_by_product"] += 1
    ws.left_norm = LeftNorm(out, weight, eps, h, sums, blocks)
    ws.counts["norms_left"] += 1
    return True


def gemm(out, a, w, accumulate, M, N, K, lda, ldw, ldc, may_defer=False, ws: Optional[KernelWorkspace] = None,
         left: Optional[LeftNorm] = None, next_norm=None, whole: bool = False) -> bool:
    if not _gemm_ok(a, w, K, lda, ldw):
        return False
    if accumulate:
        epilogue = EPI_ACCUM
    elif out.dtype == torch.bfloat16:
        epilogue = EPI_BF16
    elif out.dtype == torch.float32:
        epilogue = EPI_F32
    else:
        return False
    if left is not None:
        return _rows(out.data_ptr(), epilogue, ldc, a, w, M, N, K, lda, ldw, ws, left)
    may_defer = may_defer and ws is not None      # pieces can only wait in a workspace that outlives the call
    if M > SKINNY_MAX_ROWS:
        # few output tiles, long k: split k so that every compute unit has work; the pieces
        # stay in the workspace for the next norm of this stream
        splits = _tile_splits(M, N, K) if may_defer else 1
        if splits > 1:
            ws.pending = PendingUpdate(out, _tiles_in_pieces(a, w, M, N, K, lda, ldw, splits, ws), accumulate)
            ws.counts["deferred"] += 1
            return True
        _lib.call("bf16", "pi_gemm_mfma", out.data_ptr(), epilogue, ldc, a.data_ptr(), lda, w.data_ptr(), ldw, M, N, K, 1,
                  _tile_shape(M, N, K, 1), _stream())
        return True
    splits = _skinny_splits(M, N, K) if lda < RING_MAX_STRIDE > ldw else _far_rows_splits(M, N, K)
    if may_defer and accumulate and splits > 1 and next_norm is not None and _finish(out, a, w, M, N, K, lda, ldw, next_norm, ws):
        return True
    if whole and splits > 1 and not may_defer and M <= FEW_TOKENS and K <= FEW_TOKENS_WHOLE_K and _rows(out.data_ptr(), epilogue, ldc, a, w, M, N, K, lda, ldw, ws):
        return True
    pieces = _skinny(out.data_ptr(), epilogue, ldc, a, w, M, N, K, lda, ldw, splits, ws)
    if pieces is not None:
        if may_defer:
            ws.pending = PendingUpdate(out, pieces, accumulate)          # the next norm of this stream adds them
            ws.counts["deferred"] += 1
        else:
            _lib.call("core", "pi_splitk_reduce", out.data_ptr(), epilogue, ldc, pieces.part.data_ptr(), pieces.splits,
                      M, N, _stream())
    return True


def _float32_ok(a, w, K, lda, ldw) -> bool:
    return (K % 4 == 0 and lda % 4 == 0 and ldw % 4 == 0 and a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and max(lda, ldw) < FLOAT32_MAX_STRIDE)


def _general_streams_faster(M: int, N: int, K: int) -> bool:
    """Products of so few rows that the vector unit keeps up with the memory: the general kernel's form for them then streams the
    weights faster.  One or two rows from k = 512 on (N x K, one row, general and matrix-core kernel: 2,048 x 2,048 8.0 and 9.5 us,
    512 x 2,048 6.7 and 9.4, 16,384 x 4,096 50 and 68, 16,384 x 2,048 27.7 and 28.3; 4,096 x 256 6.6 and 4.6); up to eight rows of
    long k in a matrix of many rows (four rows of 8,192 x 8,192 68 and 80, of 8,192 x 4,096 39 and 32)."""
    return (M <= 2 and K > 512) or (M <= 8 and K >= 8192 and N >= 8192)


def _float32_product(out, a, w, accumulate, M, N, K, lda, ldw, ldc, ws: Optional[KernelWorkspace], read_by_next: bool) -> Optional[Partials]:
    """Run the float32 matrix-core product; returns the pieces when k was cut (then ``out`` is not touched)."""
    made = _lib.load("core").pi_gemm_float32_pieces(M, N, K, GEMM_PART_FLOATS, read_by_next)
    buf = _piece_buffer(ws, made * M * N, a.device) if made > 1 else None
    if out is None and buf is None:
        return None                       # pieces were wanted, and it makes none
    _lib.call("core", "pi_gemm_float32", None if out is None else out.data_ptr(), ldc, a.data_ptr(), lda, w.data_ptr(), ldw, M, N, K, int(accumulate),
              None if buf is None else buf.data_ptr(), GEMM_PART_FLOATS if buf is not None else 0, read_by_next, _stream())
    if buf is None:
        return None
    if ws is not None:
        ws.float32_counts["split_products"] += 1
    return Partials(buf, made, M, N, of_float32=True)


def gemm_float32(out, a, w, accumulate, M, N, K, lda, ldw, ldc, may_defer=False, ws: Optional[KernelWorkspace] = None) -> bool:
    """out (+)= a @ w^T, all float32, by the float32 matrix-core kernels; what a product of few tiles leaves in pieces is
    left to the stream's next reader (an update, ``may_defer``) or added at once."""
    if not _float32_ok(a, w, K, lda, ldw) or _general_streams_faster(M, N, K):
        return False
    may_defer = may_defer and accumulate and ws is not None       # a result that is written, not added, is whole when the call returns
    pieces = _float32_product(out, a, w, accumulate, M, N, K, lda, ldw, ldc, ws, may_defer)
    if pieces is not None and may_defer:
        ws.pending = PendingUpdate(out, pieces, accumulate)
        ws.float32_counts["deferred"] += 1
    elif pieces is not None:
        _lib.call("core", "pi_splitk_reduce", out.data_ptr(), EPI_ACCUM if accumulate else EPI_F32, ldc, pieces.part.data_ptr(), pieces.splits, M, N, _stream())
    return True


def gemm_float32_pieces(a, w, ws: Optional[KernelWorkspace]) -> Optional[Partials]:
    """a @ w^T in float32 left in pieces in the workspace, if this product is one whose k-range is cut."""
    if ws is None:
        return None
    M, K = a.shape
    N = w.shape[0]
    lda, ldw = a.stride(0) if M > 1 else K, w.stride(0)
    if a.stride(1) != 1 or w.stride(1) != 1 or not _float32_ok(a, w, K, lda, ldw) or _general_streams_faster(M, N, K):
        return None
    return _float32_product(None, a, w, False, M, N, K, lda, ldw, N, ws, True)


@functools.lru_cache(maxsize=4096)
def float32_gate_in_product(M: int, N: int, K: int, units: int) -> bool:
    """Whether a gated float32 product (N = 2I rows of weights) applies its unit before anything is stored, which needs whole
    sums, or leaves it to a kernel of its own behind a product whose k may be cut.  More than 32 rows: where the product would
    not be cut anyway (64 rows, 1,024 features, k 4,096: 85 us whole, 21 in eight pieces with the unit).  Fewer rows stream the
    weights in blocks of 32 rows: in the product where these nearly are as many as the units (16 rows, 3,072 features, k 2,048:
    16 and 21 us), or where k is short (8 rows, 512 features, k 512: 7.0 and 7.2; 32 rows, 1,024 features, k 4,096: 31 and 23).
    One or two rows, which the general kernel streams faster: up to k of 2,048 (8,192 features, one row: 26.9 and 28.8 us, at
    3,072 39.5 and 39.6, at 4,096 69 and 51), with few features to 1,024 (2,048 features: 9.0 and 10.0; 256: 8.6 and 7.0)."""
    if M > FLOAT32_ROWS:
        return _lib.load("core").pi_gemm_float32_pieces(M, N, K, GEMM_PART_FLOATS, 2) == 1
    blocks, general = N // 32, _general_streams_faster(M, N, K)
    if 4 * blocks >= 3 * units:
        return K <= 2048 or not general
    if general:
        return K <= 1024 and 8 * blocks >= 3 * units
    return K <= 1024 if M <= 16 else K <= 512 and 8 * blocks >= units


def gemm_swiglu_float32(out, a, w, M, N, K, lda, ldw) -> bool:
    """``w`` [N = 2I, K] with gate / up rows interleaved in blocks of 16; out [M, I], all float32."""
    if not _float32_ok(a, w, K, lda, ldw) or N % 32 or not float32_gate_in_product(M, N, K, compute_units()):
        return False
    _lib.call("core", "pi_gemm_float32_swiglu", out.data_ptr(), out.stride(0), a.data_ptr(), lda, w.data_ptr(), ldw, M, N, K, _stream())
    return True


RANGES_MAX_TOKENS = 16      # the weight-streaming kernel merges key ranges on the way in for up to this many tokens
RANGES_HEAD_DIM_STEP = 64   # ... of heads whose size is a multiple of its k step
# ... and for weights up to this size: the merging kernel has 64 weight rows per block, half the
# blocks of the plain one, which a larger matrix needs to stream at full rate (measured, batch 1
# to 16 at context 4,096: 8.4 MB 1 to 3 % faster per step, 19 MB and 34 MB 2 to 6 % slower)
RANGES_MAX_WEIGHT_BYTES = 12 << 20


def ranges_product_ok(tokens: int, head_dim: int, weight_bytes: int = 0) -> bool:
    return tokens <= RANGES_MAX_TOKENS and head_dim % RANGES_HEAD_DIM_STEP == 0 and weight_bytes <= RANGES_MAX_WEIGHT_BYTES


def merge_ranges(out: torch.Tensor, kr: KeyRanges) -> None:
    """The merged attention output, bfloat16 [tokens, heads * head_dim], by the merging kernel."""
    _lib.call("bf16", "pi_attention_combine_rows", out.data_ptr(), out.stride(0), kr.rows.data_ptr(), kr.tokens,
              kr.part.data_ptr(), kr.heads, kr.head_dim, kr.count, None, None, 0, 1.0, _stream())


def gemm_from_ranges(out, kr: KeyRanges, w, accumulate, N, ldw, ldc, may_defer, ws: Optional[KernelWorkspace], next_norm=None) -> bool:
    """out (+)= merged(kr) @ w^T by the weight-streaming kernel, which merges the key ranges as it
    stages its activations; the same bits as merging first.  With ``next_norm`` by the kernel that finishes ``out`` and leaves
    the norm, if it merges as many ranges; False if it only takes them merged."""
    M, K = kr.tokens, kr.heads * kr.head_dim
    splits = _skinny_splits(M, N, K)
    if next_norm is not None and may_defer and accumulate and splits > 1 and ws is not None and w.dtype == torch.bfloat16 and w.stride(1) == 1:
        if _finish(out, kr, w, M, N, K, 0, ldw, next_norm, ws):
            return True
        if _finish_blocks(M, N, K) and _streamed(ws, w, N, K, ldw)[1]:
            return False
    if not ranges_product_ok(M, kr.head_dim, N * K * 2) or w.dtype != torch.bfloat16 or w.stride(1) != 1 or ldw % 8 or w.data_ptr() % 16:
        return False
    if accumulate:
        epilogue = EPI_ACCUM
    elif out.dtype == torch.bfloat16:
        epilogue = EPI_BF16
    elif out.dtype == torch.float32:
        epilogue = EPI_F32
    else:
        return False
    buf = _piece_buffer(ws, splits * M * N, w.device) if splits > 1 else None
    made = ctypes.c_int(0)
    w_ptr, tiled = _streamed(ws, w, N, K, ldw)
    _lib.call("bf16", "pi_gemm_skinny_ranges", out.data_ptr(), epilogue, ldc, kr.part.data_ptr(), kr.heads, kr.head_dim, kr.count,
              w_ptr, ldw, M, N, splits, None if buf is None else buf.data_ptr(), 0 if buf is None else buf.numel(),
              ctypes.addressof(made), tiled, _stream())
    if ws is not None:
        ws.counts["ranges_merged_by_product"] += 1
    if made.value > 1:
        pieces = Partials(buf, made.value, M, N)
        if ws is not None:
            ws.counts["split_products"] += 1
        if may_defer and ws is not None:
            ws.pending = PendingUpdate(out, pieces, accumulate)
            ws.counts["deferred"] += 1
        else:
            _lib.call("core", "pi_splitk_reduce", out.data_ptr(), epilogue, ldc, pieces.part.data_ptr(), pieces.splits, M, N,
                      _stream())
    return True


def keeps_float32(M: int, N: int, K: int, units: int) -> bool:
    """Whether q, k, v that no cut of k leaves in float32 pieces still go to the rotation in float32, as one piece: while
    their tiles of 128 x 128 do not outnumber the units, and for a k above 2,048 more of them in proportion (the longer the
    product takes, the less its float32 result adds).  Results of that size are rounded once, behind the rotation, whatever
    the tile plan says about pieces; larger ones, which no plan cut, are stored in bfloat16 (one float32 piece instead, product
    and rotation: 543 x 6,144 x 4,096 43.0 -> 46.0 us, 1,280 x 3,072 x 2,048 27.6 -> 31.5; 2,048 x 3,072 x 2,048 would be
    37.9 -> 42.3).  Not for 32 tokens and fewer, nor for a k too short to be cut in two."""
    return M > SHARED_FROM_TOKENS and K >= 512 and -(-M // 128) * -(-N // 128) * 2048 <= units * max(K, 2048)


def gemm_pieces(a, w, ws: Optional[KernelWorkspace], whole: bool = False, left: Optional[LeftNorm] = None) -> Optional[Partials]:
    """a @ w^T left in float32 pieces in the workspace, if this product is one whose k-range is split; with ``whole``
    also a product in one piece (memory of its own) where ``keeps_float32`` says so.  ``left``: what ``a`` is the ``h`` of."""
    if ws is None:
        return None
    M, K = a.shape
    N = w.shape[0]
    lda, ldw = a.stride(0) if M > 1 else K, w.stride(0)
    if not _gemm_ok(a, w, K, lda, ldw) or a.stride(1) != 1 or w.stride(1) != 1:
        return None
    p = None
    if left is not None:            # few tokens: one float32 piece, of memory of its own
        out = torch.empty((1, M, N), dtype=torch.float32, device=a.device)
        return Partials(out, 1, M, N) if _rows(out.data_ptr(), EPI_F32, N, a, w, M, N, K, lda, ldw, ws, left) else None
    if M > SKINNY_MAX_ROWS:
        # a prompt portion of a few hundred tokens has too few tiles for the chip: split k there
        # too, the consumer adds the pieces
        splits = _tile_splits_of(M, N, K, compute_units(), PIECES_WORTH, norm=False)
        if splits > 1:
            p = _tiles_in_pieces(a, w, M, N, K, lda, ldw, splits, ws)
    else:
        splits = _skinny_splits(M, N, K) if lda < RING_MAX_STRIDE > ldw else _far_rows_splits(M, N, K)
        if splits > 1:
            p = _skinny(0, EPI_F32, N, a, w, M, N, K, lda, ldw, splits, ws)
    if p is not None and p.splits > 1:
        return p
    if not whole or not keeps_float32(M, N, K, compute_units()):
        return None
    out = torch.empty((1, M, N), dtype=torch.float32, device=a.device)
    gemm(out[0], a, w, False, M, N, K, lda, ldw, N, ws=ws)
    return Partials(out, 1, M, N)


EPI_GATE = 7
EPI_OF_ACTIVATION = {"relu2": 5, "gelu": 6}


def gemm_activation(out, a, w, activation, M, N, K, lda, ldw) -> bool:
    """out [M, N] bfloat16 = activation(a @ w^T) as the tile product's epilogue; only for more rows than the
    weight-streaming products take (those have no such epilogue)."""
    if not _gemm_ok(a, w, K, lda, ldw) or M <= SKINNY_MAX_ROWS:
        return False
    _lib.call("bf16", "pi_gemm_mfma", out.data_ptr(), EPI_OF_ACTIVATION[activation], out.stride(0), a.data_ptr(), lda, w.data_ptr(), ldw, M, N, K, 1,
              _tile_shape(M, N, K, 1), _stream())
    return True


def gemm_swiglu(out, a, w, M, N, K, lda, ldw, ws: Optional[KernelWorkspace] = None, left: Optional[LeftNorm] = None) -> bool:
    """``w`` [N = 2I, K] with gate / up rows interleaved in blocks of 16; out [M, I] bfloat16."""
    if not _gemm_ok(a, w, K, lda, ldw) or N % 32 or out.dtype != torch.bfloat16:
        return False
    if left is not None:
        return _rows(out.data_ptr(), EPI_SWIGLU, out.stride(0), a, w, M, N, K, lda, ldw, ws, left)
    if M > SKINNY_MAX_ROWS:
        _lib.call("bf16", "pi_gemm_mfma", out.data_ptr(), EPI_SWIGLU, out.stride(0), a.data_ptr(), lda, w.data_ptr(), ldw,
                  M, N, K, 1, _tile_shape(M, N, K, 1), _stream())
    else:
        _skinny(out.data_ptr(), EPI_SWIGLU, out.stride(0), a, w, M, N, K, lda, ldw, 1, ws, pieces_ws=False)
    return True


def gemm_clamped_glu(out, a, w, bias, limit, alpha, M, N, K, lda, ldw) -> bool:
    """``w`` [N = 2I, K] and ``bias`` (float32 [N]) with gate / up rows interleaved in blocks of 16; out [M, I]
    bfloat16 gets the clamped gated unit of the products.  The tile kernels only: steps of more rows than the
    weight-streaming kernels take."""
    if not _gemm_ok(a, w, K, lda, ldw) or N % 32 or out.dtype != torch.bfloat16 or M <= SKINNY_MAX_ROWS:
        return False
    _lib.call("bf16", "pi_gemm_mfma_clamped_glu", out.data_ptr(), out.stride(0), a.data_ptr(), lda, w.data_ptr(), ldw, M, N, K,
              bias.data_ptr(), float(limit), float(alpha), _tile_shape(M, N, K, 1), _stream())
    return True


def clamped_mlp(x, act, a, w_gate_up, bias, limit, alpha, w_down, x_bias, next_norm, ws: KernelWorkspace, left: Optional[LeftNorm]) -> bool:
    """A clamped gated feed-forward of a few tokens as two kernels: the unit (``act``) in the gate | up product, and the down
    product with its bias finishing the stream ``x`` and leaving its next norm.  False, and nothing done, for what these do not take."""
    M, I = act.shape
    K, N = a.shape[1], x.shape[1]
    lda = a.stride(0) if M > 1 else K
    if (M > FEW_TOKENS or not _gemm_ok(a, w_gate_up, K, lda, K) or not ws.has_stream_copy(w_gate_up) or not ws.has_stream_copy(w_down) or I % 16
            or max(lda, K, I) >= RING_MAX_STRIDE or _skinny_splits(M, N, I) < 2 or not _finish_blocks(M, N, I) or next_norm[0].numel() != N or not next_norm[0].is_contiguous()):
        return False
    w_ptr, _ = _streamed(ws, w_gate_up, 2 * I, K, K)
    _lib.call("bf16", "pi_gemm_rows_clamped", act.data_ptr(), act.stride(0), a.data_ptr(), lda, w_ptr, M, 2 * I, K, bias.data_ptr(), float(limit), float(alpha),
              None if left is None else left.sums.data_ptr(), 0 if left is None else left.count, 0.0 if left is None else left.eps, _stream())
    ws.counts["gated_epilogues"] += 1
    if left is not None:
        ws.counts["left_norms_read"] += 1
    return _finish(x, act, w_down, M, N, I, act.stride(0), I, next_norm, ws, x_bias)


HEAD_TILES_FROM_TOKENS = 129   # a product per head takes the grouped tile kernel from this many tokens on


@functools.lru_cache(maxsize=64)
def _head_tiles(M: int, heads: int, device) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """The grouped tile kernel's list for a product per head: head h's rows are all M rows, cut into tiles of 128."""
    rows = _lib.load("bf16").pi_gemm_mfma_group_tile_rows()
    starts = np.arange(0, M, rows, dtype=np.int32)
    group = np.repeat(np.arange(heads, dtype=np.int32), len(starts))
    row0 = np.tile(starts, heads)
    count = np.minimum(rows, M - row0).astype(np.int32)
    return tuple(torch.from_numpy(x).to(device) for x in (group, row0, count))


def head_gemm(out, a, w_rows, heads: int, K: int, N: int, a_head: int, out_head: int, lda: int, ldc: int, gate=None, gate_stride: int = 0) -> bool:
    """A product per head (``w_rows`` [heads, N, K]) as one launch of the grouped tile kernel, every head a group that
    sits at columns of its own in the rows of ``a`` and ``out``; False: not for these sizes (few tokens, or heads that
    do not start at multiples of 8 columns)."""
    M = a.shape[0]
    if M < HEAD_TILES_FROM_TOKENS or K % 8 or lda % 8 or a_head % 8 or out_head % 8 or a.data_ptr() % 16 or w_rows.data_ptr() % 16:
        return False
    if 256 * lda >= (1 << 29) or ldc >= (1 << 23) or out.data_ptr() % 4:
        return False
    group, row0, count = _head_tiles(M, heads, a.device)
    _lib.call("bf16", "pi_gemm_mfma_grouped", out.data_ptr(), EPI_BF16 if gate is None else EPI_GATE, ldc, a.data_ptr(), lda, w_rows.data_ptr(), K, N * K,
              group.data_ptr(), row0.data_ptr(), count.data_ptr(), group.numel(), N, K, a_head, out_head, 0.0, 0.0,
              None if gate is None else gate.data_ptr(), gate_stride, _stream())
    return True


# ----------------------------------------------------------------------------- attention
def attention_tile_rows(num_heads: int, num_kv_heads: int, head_dim: int) -> int:
    return _lib.load("bf16").pi_attention_tile_rows(num_heads, num_kv_heads, head_dim)


def attention_blocks_per_unit(head_dim: int) -> int:
    """Blocks of the tile kernel that one compute unit holds at a time: two up to head size 64,
    one above (its LDS and registers).  More seats than that only queue behind the first and
    leave the deal of tiles to blocks uneven: at head size 128 a 2,048-token prompt took 104 us
    with two seats per unit and 84 us with one."""
    return 2 if head_dim <= 64 else 1


def deal_tiles(walks: List[int], seats: int) -> np.ndarray:
    """[rounds, seats] tile indices (-1: none): the tiles sorted by the keys they walk, longest first, a round at a time, and
    in every round the longest to the block that has least so far.  The blocks' sums then differ by no more than the longest
    and the shortest tile of one round (a seat left empty counts as a tile of nothing).  Dealt back and forth without a look
    at the sums, a last round that is not full fell to the blocks with the longest tiles: two prompts of 1,501 and 1,126
    tokens in tiles of four on 256 blocks ended with 36 rounds of keys in the longest block instead of 32, 28 in the mean
    (heads of 256: 142 us, now 132)."""
    work = np.asarray(walks, np.int64)
    by_work = np.argsort(-work, kind="stable")
    rounds = -(-len(by_work) // seats)
    if rounds == 1:
        order = np.full((1, seats), -1, np.int32)
        order[0, :len(by_work)] = by_work
        return order
    order, dealt = np.full((rounds, seats), -1, np.int32), np.zeros(seats, np.int64)
    for k in range(rounds):
        part = by_work[k * seats:(k + 1) * seats]
        cols = np.argsort(dealt, kind="stable")[:len(part)]
        order[k, cols] = part
        dealt[cols] += work[part]
    return order


@dataclass(frozen=True)
class AttentionPlanner:
    """Makes a step's work lists for the prompt-attention tile kernel.  Mixers whose planners are
    equal (same tile height, window, kv heads) share one plan per step.  ``plan`` runs on the
    host before the step's metadata is uploaded; its arrays ride in that one copy."""

    tile_rows: int            # query rows of a tile (the kernel's, for these head counts)
    window: int               # 0: all keys
    num_kv_heads: int
    singles_apart: bool       # requests that bring one token go to the key-split kernel instead
    units: int                # compute units of the device
    blocks_per_unit: int = 2  # blocks that a unit holds at a time (attention_blocks_per_unit)
    chunk: int = 0            # C > 0: a token sees the keys of its own chunk of C positions only
    keep: int = 0             # N > 0: a token sees the first N keys besides

    def plan(self, q_lens: Sequence[int], kv_lens: Sequence[int]):
        """None for a step of single tokens only (the key-split kernel needs no list); otherwise
        (int32 host arrays by name, a function from their device views to a ``TilePlan``)."""
        if self.singles_apart and all(n == 1 for n in q_lens):
            return None
        tile_rows, window, chunk = self.tile_rows, self.window, self.chunk
        singles = tuple(r for r, n in enumerate(q_lens) if n == 1) if self.singles_apart else ()
        if len(singles) == len(q_lens):
            singles = ()
        skipped = set(singles)
        req, q0, walks, first_row, n_tok = [], [], [], [], []
        row0 = 0
        for r, (n, kv) in enumerate(zip(q_lens, kv_lens)):
            if r not in skipped:
                for start in range(0, n, tile_rows):
                    req.append(r)
                    q0.append(start)
                    first = kv - n + start                         # position of the tile's first token
                    last = first + min(tile_rows, n - start) - 1
                    lo = max(0, first - window + 1) if window > 0 else 0
                    if chunk > 0:
                        lo = max(lo, first - first % chunk)
                    walks.append(last // 128 - lo // 128 + 1 + min(-(-self.keep // 128), lo // 128))
                    first_row.append(row0 + start)
                    n_tok.append(min(tile_rows, n - start))
            row0 += n
        seats_wanted = max(1, self.blocks_per_unit * self.units // max(1, self.num_kv_heads))
        # too few tiles for the chip (a portion of a few hundred tokens): cut the key range of
        # the long ones into equal shares; the shares' partial results are merged afterwards
        cuts = cut_count(walks, seats_wanted)
        t_req, t_q0, t_cut, t_z0, t_walk, rows = [], [], [], [], [], []
        for i in range(len(req)):
            k = cuts if cuts > 1 and walks[i] >= 2 * cuts else 1
            z0 = len(rows) if k > 1 else 0
            if k > 1:
                rows.extend(range(first_row[i], first_row[i] + n_tok[i]))
            for c in range(k):
                t_req.append(req[i]); t_q0.append(q0[i]); t_cut.append(c | (k << 8)); t_z0.append(z0)
                t_walk.append(-(-walks[i] // k))
        seats = max(1, min(len(t_req), seats_wanted))
        order = deal_tiles(t_walk, seats)
        arrays = {"req": np.asarray(t_req, np.int32), "q0": np.asarray(t_q0, np.int32), "cut": np.asarray(t_cut, np.int32),
                  "z0": np.asarray(t_z0, np.int32), "rows": np.asarray(rows, np.int32), "order": order.reshape(-1),
                  "singles": np.asarray(singles, np.int32)}
        z, rounds = len(rows), order.shape[0]
        longest_single = max((kv_lens[r] for r in singles), default=0)
        singles_uneven = lengths_uneven([kv_lens[r] for r in singles])

        def finish(views: Dict[str, torch.Tensor]) -> "TilePlan":
            return TilePlan(req=views["req"], q0=views["q0"], cut=views["cut"], z0=views["z0"], rows=views["rows"],
                            cut_tokens=z, cuts=cuts if z else 1, order=views["order"], rounds=rounds, seats=seats,
                            singles=singles, single_ids=views["singles"], longest_single=longest_single, singles_uneven=singles_uneven)

        return arrays, finish


@functools.lru_cache(maxsize=None)
def attention_planner(dtype, num_heads: int, num_kv_heads: int, head_dim: int, page_size: int, window: int,
                      device, chunk: int = 0, keep: int = 0) -> Optional[AttentionPlanner]:
    """The planner for a mixer of these sizes, or None when the general kernel serves it."""
    if dtype != torch.bfloat16 or head_dim not in TILE_HEAD_DIMS or page_size % 16:
        return None
    tile_rows = attention_tile_rows(num_heads, num_kv_heads, head_dim)
    if tile_rows < 1:
        return None
    units = torch.cuda.get_device_properties(device).multi_processor_count
    return AttentionPlanner(tile_rows, int(window), num_kv_heads, num_heads // num_kv_heads <= 16, units,
                            attention_blocks_per_unit(head_dim), int(chunk), int(keep))


def upload_arrays(arrays: Dict[str, np.ndarray], device) -> Dict[str, torch.Tensor]:
    """Concatenate int32 arrays (each padded to 16 bytes), copy once, return device views."""
    offsets, total = {}, 0
    for name, arr in arrays.items():
        offsets[name] = (total, arr.size)
        total += (arr.size + 3) // 4 * 4
    packed = np.zeros(max(total, 4), np.int32)
    for name, arr in arrays.items():
        o, n = offsets[name]
        packed[o:o + n] = arr.reshape(-1)
    dev = torch.from_numpy(packed).to(device)
    return {name: dev[o:o + n] for name, (o, n) in offsets.items()}


def _tile_plan(ctx, planner: AttentionPlanner, device) -> "TilePlan":
    """The step's plan: the one the step function uploaded with its metadata, or - for a caller
    that made its context by hand - one made and uploaded here."""
    plans = getattr(ctx, "plans", None)
    if plans is None:
        plans = ctx.plans = {}
    plan = plans.get(planner)
    if plan is None:
        arrays, finish = planner.plan(ctx.q_lens, ctx.kv_lens)
        plan = plans[planner] = finish(upload_arrays(arrays, device))
    return plan


@dataclass
class TilePlan:
    """A step's work list for the tile kernel (device int32 arrays, one entry per tile or per
    share of a cut tile)."""

    req: torch.Tensor          # the entry's request
    q0: torch.Tensor           # its first token among the request's tokens of this step
    cut: torch.Tensor          # share | shares << 8 of the tile's key range
    z0: torch.Tensor           # first row of the tile in ``rows`` (cut tiles only)
    rows: torch.Tensor         # token rows of the cut tiles, in the order of their partial results
    cut_tokens: int
    cuts: int                  # shares per cut tile (the same for all of a step)
    order: torch.Tensor        # [rounds, seats]: which entry a block takes in which round (-1: none)
    rounds: int
    seats: int
    singles: Tuple[int, ...] = ()             # requests that bring one token beside requests that bring more
    single_ids: Optional[torch.Tensor] = None  # the same on the device
    longest_single: int = 0                   # the longest context among them
    singles_uneven: bool = False              # their contexts are uneven (lengths_uneven)


MAX_TILE_CUTS = 8
MIN_ROUNDS_PER_SHARE = 4       # a share of a cut tile walks at least this many rounds of 128 keys ...
MIN_ROUNDS_SAVED = 6           # ... and the cut shortens the longest walk by at least this many


def cut_count(walks: List[int], seats_wanted: int) -> int:
    """In how many shares the key range of a step's long tiles is cut: 1 unless the tiles are
    fewer than half the blocks the chip holds; then as many as fill it, while a share keeps
    enough rounds of 128 keys to be worth an entry of its own (its queries loaded again, its
    partial result written and merged: about the time of six rounds).  Measured at head sizes
    64 and 128, 64 to 1,024 tokens ending at 256 to 8,192: shares of two rounds made 256 tokens
    at 2,048 slower than uncut (56 us against 46; with shares of four 29 us), and two shares of
    a walk of eight rounds or less never paid."""
    tiles = len(walks)
    if tiles == 0 or tiles * 2 > seats_wanted:
        return 1
    longest = max(walks)
    cuts = min(MAX_TILE_CUTS, seats_wanted // tiles, longest // MIN_ROUNDS_PER_SHARE)
    if cuts < 2 or longest - -(-longest // cuts) < MIN_ROUNDS_SAVED:
        return 1
    return cuts


def decode_length_bucket(max_kv_len: int) -> int:
    """The power of two (at least one key range's worth) that a decode step's longest context
    is rounded up to.  Key ranges are chosen per bucket, so a step gives the same numbers
    whether it runs eagerly or replays the graph captured for its bucket."""
    bucket = DECODE_MIN_KEYS_PER_SPLIT
    while bucket < max_kv_len:
        bucket *= 2
    return bucket


def decode_splits(R: int, num_kv_heads: int, max_kv_len: int) -> int:
    """Key ranges per (request, kv head): enough waves to fill the chip, no more than the
    keys of the step's length bucket are worth."""
    splits = max(1, min(MAX_DECODE_SPLITS, -(-DECODE_WAVES_PER_UNIT * compute_units() // (R * num_kv_heads))))
    return min(splits, max(1, decode_length_bucket(max_kv_len) // DECODE_MIN_KEYS_PER_SPLIT))


def decode_block_waves(splits: int, R: int, num_kv_heads: int, max_kv_len: int, head_dim: int = 64) -> int:
    """Waves per block of the decode attention, which share a request's keys of one kv head and merge in the block: they take
    the place of ``splits`` ranges (more than 1: one range then, and no merging kernel), or 1.  Where there are no ranges to
    replace they are worth it for lengths that are uneven only (``_uneven_lengths``).  Steps whose ranges the next
    product may merge keep them."""
    blocks, bucket = R * num_kv_heads, decode_length_bucket(max_kv_len)
    rounds = -(-blocks // compute_units())
    fill = DECODE_WAVES_FILL_LONG if rounds > 1 and bucket > DECODE_WAVES_LONG else DECODE_WAVES_FILL
    if R <= RANGES_MAX_TOKENS or splits > 4 or blocks < fill * rounds * compute_units():
        return 1
    if splits > 1:
        return 2 if splits == 2 else 4
    return 2 if rounds < 3 and bucket > DECODE_WAVES_MIN_KEYS * max(1, head_dim // 64) else 1


def decode_range_waves(splits: int, R: int, num_kv_heads: int) -> Tuple[int, int]:
    """(ranges, waves that share one) in place of ``splits`` ranges of a wave each: whoever merges them has half as many, which
    steps of up to four requests gain by, as long as the blocks are one round over the units.  Decode steps with ranges of a
    wave each and of two, us, going on from so many keys: 1B sizes, one request of 4,000 and 16,000 850 / 804 and 906 / 868, two of
    2,000 809 / 795, four of 1,000 and 4,000 811 / 803 and 851 / 842; 8B sizes, one of 4,000 1,000 / 976, two of 4,000 1,026 / 1,017,
    four of 8,000 1,104 / 1,102.  264 or 288 blocks: three of 8,000 907 / 922, six and eleven of 1,000 840 / 840 and 931 / 943, twelve
    of 4,000 1,139 / 1,175.  256 blocks, more requests: eight of 4,000 971 / 974, sixteen 1,233 / 1,245."""
    ranges = -(-splits // 2)
    if R <= RANGES_SHARED_UP_TO and R * splits >= RANGES_TO_SHARE and R * ranges * num_kv_heads <= compute_units():
        return ranges, 2
    return splits, 1


def lengths_uneven(kv_lens) -> bool:
    """Whether a step's contexts differ enough for waves that share one: the longest against the mean."""
    if len(kv_lens) <= RANGES_MAX_TOKENS:
        return False
    lens = np.asarray(kv_lens)
    return int(lens.max()) * len(lens) > UNEVEN * int(lens.sum())


def _waves_or_ranges(ctx, splits: int, R: int, num_kv_heads: int, head_dim: int, longest: int, bound: int, plan=None,
                     plain: bool = True) -> Tuple[int, int, Optional[int]]:
    """(ranges, waves, where the device reads whether the waves are to share at all) of a decode attention; ``bound`` > 0: a
    token sees so many keys at most; ``plain``: heads without options; ``plan``: the requests are the single tokens of a step with portions, which the host knows."""
    bounded = 0 < bound < decode_length_bucket(longest)
    waves = decode_block_waves(splits, R, num_kv_heads, min(longest, bound) if bounded else longest, head_dim)
    if waves == 1 or splits > 1:
        if waves > 1:
            return 1, waves, None
        # as the kernel that starts from the projection, to the same bits
        return (*(decode_range_waves(splits, R, num_kv_heads) if plain and head_dim in FUSED_DECODE_HEAD_DIMS else (splits, 1)), None)
    if bounded:                                       # the contexts' lengths do not say how many keys are seen
        return 1, 1, None
    if plan is not None:
        return 1, waves if plan.singles_uneven else 1, None
    flag = getattr(ctx, "uneven", None)
    return (1, 1, None) if flag is None else (1, waves, flag.data_ptr())


def _attn_part(ws: Optional[KernelWorkspace], floats: int, device) -> torch.Tensor:
    return ws.attn_part if ws is not None else torch.empty(max(4, floats), dtype=torch.float32, device=device)


def _decode_splits_that_fit(ws, n_req: int, num_heads: int, num_kv_heads: int, head_dim: int, longest: int) -> int:
    splits = decode_splits(n_req, num_kv_heads, longest)
    if ws is not None:
        while splits > 1 and n_req * num_heads * splits * (head_dim + 4) > ws.attn_part.numel():
            splits -= 1
    return splits


def paged_attention(out, q, k_cache, v_cache, block_table, ctx, num_heads, num_kv_heads, head_dim,
                    page_size, scale, window, pages, ws: Optional[KernelWorkspace] = None, slopes=None, sinks=None, gate=None,
                    softcap: float = 0.0, out_scale: float = 1.0, chunk: int = 0, gate_stride: int = 0, keep: int = 0) -> bool:
    """``slopes`` / ``sinks`` (float32 [heads]) and ``gate`` (float32 [tokens, heads]; with ``gate_stride`` rows of one
    unactivated gate per feature): a distance bias, a sink in the softmax and an output gate per head (None: none); ``softcap`` > 0: scaled scores s become
    softcap * tanh(s / softcap); ``out_scale``: a factor on every output; ``keep`` > 0: the first so many keys are seen besides."""
    opt = tuple(None if t is None else t.data_ptr() for t in (slopes, sinks, gate)) + (int(gate_stride), float(softcap), float(out_scale), int(chunk), int(keep))
    if head_dim not in DECODE_HEAD_DIMS or page_size % 16 or q.data_ptr() % 16 or q.stride(0) % 8 or out.stride(0) % 4:
        return False
    if gate_stride and (gate_stride % 4 or gate.data_ptr() % 16):
        return False
    G = num_heads // num_kv_heads
    R = ctx.R

    def decode_kernel(n_req: int, req_ids: int, longest: int, plan=None) -> None:
        # (a token's keys end at its chunk's start, whatever the context)
        splits = _decode_splits_that_fit(ws, n_req, num_heads, num_kv_heads, head_dim, min(longest, chunk + keep) if chunk else longest)
        bound = min(window or 1 << 30, chunk + keep if chunk else 1 << 30) if window or chunk else 0
        splits, waves, uneven = _waves_or_ranges(ctx, splits, n_req, num_kv_heads, head_dim, longest, bound, plan, opt == PLAIN_HEADS)
        part = _attn_part(ws, n_req * num_heads * splits * (head_dim + 4), q.device)
        _lib.call("bf16", "pi_attention_decode", out.data_ptr(), out.stride(0), q.data_ptr(), q.stride(0),
                  k_cache.data_ptr(), v_cache.data_ptr(), block_table.data_ptr(), block_table.shape[1],
                  ctx.q_start.data_ptr(), ctx.kv_len.data_ptr(), req_ids, n_req, num_heads, num_kv_heads, head_dim,
                  page_size, float(scale), int(window), pages, splits, waves, uneven, part.data_ptr(), part.numel(), *opt, _stream())

    if ctx.all_decode and G <= 16:
        decode_kernel(R, 0, ctx.max_kv_len)
        return True
    planner = attention_planner(q.dtype, num_heads, num_kv_heads, head_dim, page_size, window, q.device, int(chunk), int(keep))
    if planner is None:
        return False
    # A step of prompt portions and single tokens: the single tokens, whose keys no other token
    # of the step shares, go to the key-split kernel (a tile of one token would walk its whole
    # context in one block, mostly on padding); the portions go to the tile kernel.
    plan = _tile_plan(ctx, planner, q.device)
    if plan.singles:
        decode_kernel(len(plan.singles), plan.single_ids.data_ptr(), plan.longest_single, plan)
    floats = plan.cut_tokens * num_heads * plan.cuts * (head_dim + 4)
    tile_part = ws.tile_part_for(floats) if ws is not None else torch.empty(max(4, floats), dtype=torch.float32, device=q.device)
    _lib.call("bf16", "pi_attention_prefill_mfma", out.data_ptr(), out.stride(0), q.data_ptr(), q.stride(0),
              k_cache.data_ptr(), v_cache.data_ptr(), block_table.data_ptr(), block_table.shape[1],
              ctx.q_start.data_ptr(), ctx.kv_len.data_ptr(), plan.req.data_ptr(), plan.q0.data_ptr(), plan.cut.data_ptr(),
              plan.z0.data_ptr(), tile_part.data_ptr(), plan.order.data_ptr(), plan.rounds, plan.seats, num_heads,
              num_kv_heads, head_dim, page_size, float(scale), int(window), pages, *opt, _stream())
    if plan.cut_tokens:
        _lib.call("bf16", "pi_attention_combine_rows", out.data_ptr(), out.stride(0), plan.rows.data_ptr(), plan.cut_tokens,
                  tile_part.data_ptr(), num_heads, head_dim, plan.cuts, opt[1], opt[2], opt[3], opt[5], _stream())
    return True


def float32_attention_us(q_lens, kv_lens, num_heads: int, num_kv_heads: int, head_dim: int, tile_tokens: int, reach: int = 0) -> Tuple[float, float]:
    """What a step takes on the float32 path's tile kernel and on its general kernel (``reach`` > 0: a token sees at most so many
    keys).  Tiles: a block walks its keys 64 at a time, whether its 64 rows of (token, head) are there or not; the longest
    walk, or all of them dealt over the chip.  General: a wave per token and head, so its (query, key) pairs, and the chain
    along the longest context, cut into ranges where the waves are few.  Fitted to 400 random steps on an MI355X - prompts,
    portions over up to 12,000 keys, single tokens beside them; heads of 16 to 128, 1 to 12 per kv head; windows - where each
    kernel is the faster one in about half, by up to 9 times."""
    units, seen = compute_units(), reach or 1 << 30
    rounds, longest, pairs, chain = 0.0, 0.0, 0.0, 0
    for n, kv in zip(q_lens, kv_lens):
        before, rows = kv - n, min(tile_tokens, n)
        rounds += -(-n // tile_tokens) * (min(before + (n + rows) / 2, seen + rows) / 64 + 0.5)
        longest = max(longest, -(-min(kv, seen + tile_tokens) // 64))
        pairs += n * min(before + n / 2, seen)
        chain = max(chain, min(kv, seen))
    blocks_per_tile = num_heads * tile_tokens // 64
    tiles = 5.3 + (1.2 + 0.053 * head_dim) * max(longest, rounds * blocks_per_tile / units)
    if chain >= 256:
        chain /= max(1, min(64, 4096 // (sum(q_lens) * num_heads)))
    return tiles, 8.3 + pairs * num_heads * head_dim * 0.9e-6 + chain * (0.078 + 0.0002 * head_dim)


# What the tile kernel must promise at most of the general kernel's time, for both are off by a fifth in places.  Of the 400
# steps above 13 then take more than 3 % longer than on the general kernel (by a few microseconds), and the mean is 2.3 % above
# the better of the two; with the tile kernel from 32 tokens on (the rule before) it was 121 steps and 15 %: 32 tokens at 32,768
# keys, 24 heads of 128: 3,600 us, 2,450 now; 31 single tokens and 33 at 2,000: 590 us, 450 now.
FLOAT32_TILES_WORTH = 0.8


def paged_attention_float32(out, q, k_cache, v_cache, block_table, ctx, num_heads, num_kv_heads, head_dim, page_size, scale, window, pages,
                            slopes=None, sinks=None, gate=None, softcap: float = 0.0, out_scale: float = 1.0, chunk: int = 0,
                            gate_stride: int = 0) -> bool:
    """Prompt portions on the float32 path, by the matrix-core tile kernel (options as for ``paged_attention``)."""
    if (head_dim % 16 or head_dim > 128 or page_size % 16 or q.data_ptr() % 16 or out.data_ptr() % 16 or q.stride(0) % 4 or out.stride(0) % 4
            or k_cache.data_ptr() % 16 or v_cache.data_ptr() % 16):
        return False
    rows = _lib.load("core").pi_attention_float32_tile_tokens(num_heads, num_kv_heads)
    reach = min(window or 1 << 30, chunk or 1 << 30) if window or chunk else 0
    key = ("float32 attention", num_heads, num_kv_heads, head_dim, reach)
    plans = getattr(ctx, "plans", None)
    if plans is None:
        plans = ctx.plans = {}
    if key not in plans:
        tiles_us, general_us = float32_attention_us(ctx.q_lens, ctx.kv_lens, num_heads, num_kv_heads, head_dim, rows, reach)
        plans[key] = tiles_us < FLOAT32_TILES_WORTH * general_us
    if not plans[key]:
        return False
    tiles = sum(-(-n // rows) for n in ctx.q_lens)
    _lib.call("core", "pi_attention_float32", out.data_ptr(), out.stride(0), q.data_ptr(), q.stride(0), k_cache.data_ptr(), v_cache.data_ptr(),
              block_table.data_ptr(), block_table.shape[1], ctx.q_start.data_ptr(), ctx.kv_len.data_ptr(), ctx.R, tiles, num_heads, num_kv_heads,
              head_dim, page_size, float(scale), int(window), pages, None if slopes is None else slopes.data_ptr(),
              None if sinks is None else sinks.data_ptr(), None if gate is None else gate.data_ptr(), gate_stride, softcap, out_scale, chunk, _stream())
    return True


# Key ranges of the float32 decode attention: blocks per compute unit that fill the chip (32 heads on 8 kv heads of 64, 64 requests of
# 2,000 keys: 85 us with four, 105 with two; heads of 128 take registers for two: 8 requests of 2,000 34 and 43), and keys of the
# step's length bucket that a range keeps (8 requests of 600: 15.1 us with 128, 17.1 with 256), from a bucket on that is worth the
# merging kernel (one request of 150: 12.5 us in one range, 13.0 in two)
FLOAT32_DECODE_BLOCKS_PER_UNIT, FLOAT32_DECODE_MIN_KEYS, FLOAT32_DECODE_MIN_BUCKET = {64: 4, 128: 2}, 128, 512


def float32_decode_ranges(R: int, num_kv_heads: int, head_dim: int, max_kv_len: int) -> int:
    """Key ranges per request and kv head, by the step's length bucket (the same eagerly and replayed)."""
    bucket = decode_length_bucket(max_kv_len)
    if bucket < FLOAT32_DECODE_MIN_BUCKET:
        return 1
    return max(1, min(MAX_DECODE_SPLITS, FLOAT32_DECODE_BLOCKS_PER_UNIT[head_dim] * compute_units() // (R * num_kv_heads), bucket // FLOAT32_DECODE_MIN_KEYS))


def decode_attention_float32(out, qkv, ctx, table, num_heads, num_kv_heads, head_dim, k_cache, v_cache, block_table, page_size, scale, window, pages,
                             write_kv) -> bool:
    """``decode_attention_from_projection`` of the float32 path; the kernel always fills ``out``."""
    R = ctx.R
    if page_size % 16 or k_cache.data_ptr() % 16 or v_cache.data_ptr() % 16 or not _lib.load("core").pi_attention_float32_decode_takes(num_heads, num_kv_heads, head_dim):
        return False
    if not isinstance(qkv, Partials):
        if qkv.stride(1) != 1 or (R > 1 and qkv.stride(0) != qkv.shape[1]):
            return False
        qkv = Partials(qkv, 1, qkv.shape[0], qkv.shape[1])
    if qkv.M != R or qkv.N < (num_heads + (2 * num_kv_heads if write_kv else 0)) * head_dim:
        return False
    ranges = float32_decode_ranges(R, num_kv_heads, head_dim, min(ctx.max_kv_len, window) if window else ctx.max_kv_len)
    part = torch.empty(R * num_heads * ranges * (head_dim + 2), dtype=torch.float32, device=out.device) if ranges > 1 else None
    _lib.call("core", "pi_attention_float32_decode", out.data_ptr(), out.stride(0), qkv.part.data_ptr(), qkv.splits, qkv.N, R,
              None if table is None else table.data_ptr(), int(bool(write_kv)), k_cache.data_ptr(), v_cache.data_ptr(), block_table.data_ptr(),
              block_table.shape[1], ctx.q_start.data_ptr(), ctx.kv_len.data_ptr(), R, num_heads, num_kv_heads, head_dim, page_size, float(scale),
              int(window), pages, ranges, None if part is None else part.data_ptr(), 0 if part is None else part.numel(), _stream())
    return True


def decode_attention_from_projection(out, qkv, ctx, table, num_heads, num_kv_heads, head_dim, k_cache, v_cache,
                                     block_table, page_size, scale, window, pages, write_kv,
                                     ws: Optional[KernelWorkspace] = None, leave_ranges: int = 0):
    """A step of single tokens: attention straight from the q|k|v projection (``qkv``: a bfloat16
    tensor [T, N] or ``Partials``), which the kernel rotates by ``table`` (the step's cos / sin
    table [T, head_dim], or None) and whose keys and values it stores.  False: not for these sizes.
    ``leave_ranges`` (0: never; else the bytes of the weight matrix that reads the output next):
    when the keys were split into ranges and that product can merge them (``ranges_product_ok``),
    they are returned as ``KeyRanges`` and ``out`` is left alone."""
    G = num_heads // num_kv_heads
    if not ctx.all_decode or G > 16 or head_dim not in FUSED_DECODE_HEAD_DIMS or page_size % 16 or out.stride(0) % 4:
        return False
    R = ctx.R
    pieces = isinstance(qkv, Partials)
    need = (num_heads + (2 * num_kv_heads if write_kv else 0)) * head_dim
    if (qkv.M if pieces else qkv.shape[0]) != R or (qkv.N if pieces else qkv.shape[1]) < need:
        return False
    if (qkv.N % 4 or qkv.part.data_ptr() % 16) if pieces else (qkv.stride(0) % 8 or qkv.stride(1) != 1 or qkv.data_ptr() % 16):
        return False
    splits = _decode_splits_that_fit(ws, R, num_heads, num_kv_heads, head_dim, ctx.max_kv_len)
    leave = leave_ranges > 0 and ws is not None and splits > 1 and ranges_product_ok(R, head_dim, leave_ranges)
    waves, uneven = 1, None
    if leave:
        splits, waves = decode_range_waves(splits, R, num_kv_heads)
        leave = splits > 1
    else:
        splits, waves, uneven = _waves_or_ranges(ctx, splits, R, num_kv_heads, head_dim, ctx.max_kv_len, window)
    part = _attn_part(ws, R * num_heads * splits * (head_dim + 4), out.device)
    _lib.call("bf16", "pi_attention_decode_fused", out.data_ptr(), out.stride(0),
              None if pieces else qkv.data_ptr(), 0 if pieces else qkv.stride(0),
              qkv.part.data_ptr() if pieces else None, qkv.splits if pieces else 0, qkv.N if pieces else 0, R,
              None if table is None else table.data_ptr(), int(bool(write_kv)), k_cache.data_ptr(), v_cache.data_ptr(),
              block_table.data_ptr(), block_table.shape[1], ctx.q_start.data_ptr(), ctx.kv_len.data_ptr(), R, num_heads,
              num_kv_heads, head_dim, page_size, float(scale), int(window), pages, splits, waves, uneven, part.data_ptr(),
              part.numel(), int(not leave), _stream())
    if leave:
        return KeyRanges(part, splits, R, num_heads, head_dim, ctx.q_start)
    return True
