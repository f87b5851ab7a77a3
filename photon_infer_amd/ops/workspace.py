"""Scratch memory of the kernels, owned by whoever runs steps (one per ``ModelRunner``).

Nothing in this package keeps kernel state of its own.  The pieces of a product that was split
over k, the partial results of attention split over keys and the chunk records of the sampling
kernels live in a ``KernelWorkspace``; so does the one update of a residual stream that may
still be in pieces (see ``ops.gemm(..., may_defer=True)``).  Two runners have two workspaces
and never see each other's pieces; an op called without a workspace takes what it needs from
torch's allocator for that call and leaves nothing pending.
"""
from __future__ import annotations

from collections import Counter
from dataclasses import dataclass
from typing import Dict, Optional, Tuple

import torch

GEMM_PART_FLOATS = 16 << 20    # pieces of products split over k (64 MB)
ATTN_PART_FLOATS = 4 << 20     # key-split partial results of decode attention
SAMPLE_FLOATS = 1 << 18        # chunk records of the sampling kernels


@dataclass
class Partials:
    """A product [M, N] whose k-range was split: ``part`` holds float32 [splits, M, N].  ``of_float32``: the product
    of a float32 model, whose statistics are kept apart."""

    part: torch.Tensor
    splits: int
    M: int
    N: int
    of_float32: bool = False


@dataclass
class KeyRanges:
    """The attention output of a decode step (token r is request r) whose key ranges are not
    merged yet: ``part`` holds float32 [tokens, heads, count, head_dim + 4] (a range's output not
    yet normalised, then its maximum and its sum of weights).  It lives in the workspace's
    attention buffer, so it has to be consumed (``ops.gemm`` takes it as its activations) before
    the next attention of that workspace runs.  ``rows``: int32 device array, row of each token."""

    part: torch.Tensor
    count: int
    tokens: int
    heads: int
    head_dim: int
    rows: torch.Tensor

    def __bool__(self) -> bool:
        return True


@dataclass
class PendingUpdate:
    """``target += sum(pieces)`` (``accumulate`` False: ``target = sum(pieces)``, a sublayer's result that is still
    in pieces) that has not been applied yet."""

    target: torch.Tensor
    pieces: Partials
    accumulate: bool = True

    def is_for(self, x: torch.Tensor) -> bool:
        t = self.target
        return t is x or (t.data_ptr() == x.data_ptr() and t.shape == x.shape and t.stride() == x.stride())


def _version_of(x: torch.Tensor) -> Optional[int]:
    return None if x.is_inference() else x._version       # (tensors made in inference mode count no versions)


@dataclass
class LeftNorm:
    """The norm of a stream ``x`` [M, D] that the product before it made but for the root (``ops.gemm`` with ``next_norm``):
    ``h`` holds bfloat16(x * weight), ``sums`` float32 [M, count] every row's sum of x^2 in pieces.  A product that takes it
    as activations multiplies its float32 rows by 1 / sqrt(sum / D + eps).  Good until ``x`` changes: whoever writes a stream in
    place raises the tensor's version (torch's own operations do, ``ops._changes`` for the kernels).  ``count`` 0: ``h`` is
    the norm itself, whole."""

    x: torch.Tensor
    weight: torch.Tensor
    eps: float
    h: torch.Tensor
    sums: Optional[torch.Tensor]
    count: int

    def __post_init__(self):
        self.version = _version_of(self.x)

    @property
    def stale(self) -> bool:
        """The stream has been written since."""
        return _version_of(self.x) != self.version

    @property
    def shape(self):
        return self.h.shape

    @property
    def device(self):
        return self.h.device

    @property
    def dtype(self):
        return self.h.dtype

    @property
    def is_cuda(self):
        return self.h.is_cuda


def stream_layout_takes(w: torch.Tensor) -> bool:
    """Whether ``stream_layout`` has a form for ``w``."""
    return (w.dim() == 2 and w.dtype == torch.bfloat16 and w.is_contiguous() and w.shape[0] > 0 and w.shape[0] % 16 == 0
            and w.shape[1] > 0 and w.shape[1] % 64 == 0)


def stream_layout(w: torch.Tensor) -> Optional[torch.Tensor]:
    """The bfloat16 matrix ``w`` [N, K] (N a multiple of 16, K of 64, rows contiguous) as
    [N / 16][K / 64][2][4][16][8]: for every 16 rows and 64 columns, the 1 KB that a wave of the
    weight-streaming kernels loads with one instruction lies in a row (lane group g of a wave
    holds columns 16 g + 8 h .. + 7 of its row in its fragment h).  None for other matrices."""
    if not stream_layout_takes(w):
        return None
    N, K = w.shape
    tiles = w.view(N // 16, 16, K // 64, 4, 2, 8)          # [row block, row, k block, lane group, fragment, 8 columns]
    return tiles.permute(0, 2, 4, 3, 1, 5).contiguous().view(N, K)


class KernelWorkspace:
    """Buffers are made at first use and kept; ``counts`` says which paths a step took (tests
    read it: ``split_products``, ``deferred``, ``added_by_norm``, ``applied``, ``flushed``,
    ``discarded``, ``qkv_pieces``, ``ranges_merged_by_product``, ``norms_left``, ``left_norms_read``).  ``counts`` is about the 16-bit
    products; ``float32_counts`` has the same entries for pieces of float32 products."""

    def __init__(self, device):
        self.device = torch.device(device)
        self._gemm_part: Optional[torch.Tensor] = None
        self._attn_part: Optional[torch.Tensor] = None
        self._tile_part: Optional[torch.Tensor] = None
        self._sample_part: Optional[torch.Tensor] = None
        self.pending: Optional[PendingUpdate] = None
        self.left_norm: Optional[LeftNorm] = None      # what a product has made of the stream's next norm
        self.counts: Counter = Counter()
        self.float32_counts: Counter = Counter()
        # weight matrices that have a second copy in the order the weight-streaming kernels read
        # (steps of up to 128 tokens): address of the matrix -> (copy, rows, columns, the matrix
        # itself: while it is kept here, nothing else can come to lie at its address)
        self.stream_copies: Dict[int, Tuple[torch.Tensor, int, int, torch.Tensor]] = {}

    def counts_of(self, pieces: Partials) -> Counter:
        """The statistics that ``pieces`` belong to."""
        return self.float32_counts if pieces.of_float32 else self.counts

    def _buffer(self, name: str, floats: int) -> torch.Tensor:
        buf = getattr(self, name)
        if buf is None or buf.numel() < floats:
            buf = torch.empty(floats, dtype=torch.float32, device=self.device)
            setattr(self, name, buf)
        return buf

    @property
    def gemm_part(self) -> torch.Tensor:
        return self._buffer("_gemm_part", GEMM_PART_FLOATS)

    @property
    def attn_part(self) -> torch.Tensor:
        return self._buffer("_attn_part", ATTN_PART_FLOATS)

    @property
    def sample_part(self) -> torch.Tensor:
        return self._buffer("_sample_part", SAMPLE_FLOATS)

    def tile_part_for(self, floats: int) -> torch.Tensor:
        """Partial results of cut tiles, grown on demand."""
        return self._buffer("_tile_part", max(4, floats))

    def prepare(self, matrix_core_attention: bool, split_products: bool = True) -> None:
        """Make the buffers of fixed size now (before anything is captured into a graph)."""
        self.sample_part
        if split_products:
            self.gemm_part
        if matrix_core_attention:
            self.attn_part

    def add_stream_copy(self, w: torch.Tensor) -> bool:
        """Keep a copy of the bfloat16 matrix ``w`` [N, K] in the weight-streaming kernels' order
        (``stream_layout``); products of up to 128 tokens with ``w`` then read the copy.  False,
        and nothing kept, for a matrix whose sizes the layout does not take."""
        copy = stream_layout(w)
        if copy is None:
            return False
        self.stream_copies[w.data_ptr()] = (copy, w.shape[0], w.shape[1], w)
        return True

    def drop_stream_copies(self) -> None:
        """Forget every copy (their memory goes back to the allocator); products read the matrices
        themselves again.  For a caller that changes a weight matrix after load: a copy is made
        once and never refreshed."""
        self.stream_copies.clear()

    def stream_copy_of(self, w: torch.Tensor, N: int, K: int) -> Optional[torch.Tensor]:
        entry = self.stream_copies.get(w.data_ptr())
        if entry is None or entry[1] != N or entry[2] != K:
            return None
        return entry[0]

    def has_stream_copy(self, w: torch.Tensor) -> bool:
        return w.dim() == 2 and self.stream_copy_of(w, w.shape[0], w.shape[1]) is not None

    def take_left_norm(self, x: torch.Tensor, weight: torch.Tensor, eps: float) -> Optional[LeftNorm]:
        """What is left of the norm of ``x`` with these parameters, if a product has made it and ``x`` is as it was then."""
        left, self.left_norm = self.left_norm, None
        return left if left is not None and left.x is x and left.weight is weight and left.eps == eps and not left.stale else None

    def take_pending(self, x: torch.Tensor) -> Optional[Partials]:
        """The pieces still to be added to ``x``, if any; they are the caller's to add."""
        p = self.pending
        if p is not None and p.accumulate and p.is_for(x):
            self.pending = None
            return p.pieces
        return None

    def take_result(self, y: torch.Tensor) -> Optional[Partials]:
        """The pieces whose sum ``y`` is to hold, if they are still unadded (``y`` itself is then unwritten)."""
        p = self.pending
        if p is not None and not p.accumulate and p.is_for(y):
            self.pending = None
            return p.pieces
        return None
