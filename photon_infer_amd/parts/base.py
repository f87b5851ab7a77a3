"""Interfaces of the parts a layer is put together from, and their registries.

A model is data: a list of blocks, each naming a norm, a mixer, a feed-forward and an
arrangement, plus a run order.  Every part takes its sizes and constants as
constructor parameters, declares the tensors it expects (relative names) and what it
needs from the cache manager; none of them knows which model it sits in.

The reference wires one fixed block (src/arch/transformer_block.cpp:28-58: two norms,
seven matmuls, rope, mha, add, swiglu) and has no such seam; the interfaces below are
what replaces it.

Data flow convention: the residual stream ``x`` is float32 ``[T, hidden]`` in both
compute modes.  A norm reads ``x`` and writes activations ``h`` in the compute dtype;
a mixer or feed-forward reads ``h`` and *adds* its result into ``x``.
"""
from __future__ import annotations

from dataclasses import dataclass, field
from typing import Any, Callable, Dict, List, Optional, Sequence, Tuple

import torch

from .. import ops
from ..errors import UnsupportedModelError
from ..weights.loader import TensorSpec


# --------------------------------------------------------------------------- cache needs
PAGE = -1     # in a paged tensor's shape: the axis that holds a page's tokens


@dataclass(frozen=True)
class PagedTensor:
    """One tensor that a mixer keeps per token, in pages: the shape of one page of it, with ``PAGE``
    standing for the page's tokens, e.g. keys ``(kv_heads, PAGE, head_dim)``, values transposed
    ``(kv_heads, head_dim, PAGE)``, one latent vector per token ``(PAGE, width)``.  The pool is
    ``[pages, *shape]``.  ``dtype`` None: the compute dtype."""

    name: str
    shape: tuple
    dtype: Optional[torch.dtype] = None

    def page_shape(self, page_size: int) -> tuple:
        if sum(1 for d in self.shape if d == PAGE) != 1:
            raise UnsupportedModelError(f"paged tensor '{self.name}': its shape {self.shape} must name the page axis once")
        return tuple(page_size if d == PAGE else int(d) for d in self.shape)

    def page_bytes(self, page_size: int, compute_dtype: torch.dtype) -> int:
        n = 1
        for d in self.page_shape(page_size):
            n *= d
        return n * torch.empty((), dtype=self.dtype or compute_dtype).element_size()


@dataclass(frozen=True)
class PagedCacheSpec:
    """What a mixer keeps per token, in pages: any number of named tensors, each with its own
    shape and layout.  ``window`` = None keeps every token; an integer W keeps the last W
    positions, so the cache manager may hand back pages that the window has passed, and
    ``keep_first`` N keeps a sequence's first N positions besides.  Mixers with the same window and
    kept tokens share a cache group (one page pool's bookkeeping, one block table)."""

    tensors: Tuple[PagedTensor, ...]
    window: Optional[int] = None
    keep_first: int = 0


@dataclass(frozen=True)
class KVCacheSpec:
    """The usual case of ``PagedCacheSpec``: keys ``k`` [kv_heads, page, head_dim] and values
    ``v`` transposed [kv_heads, head_dim, page] (the layout the attention kernels contract in)."""

    num_kv_heads: int
    head_dim: int
    window: Optional[int] = None
    keep_first: int = 0

    @property
    def tensors(self) -> Tuple[PagedTensor, ...]:
        return (PagedTensor("k", (self.num_kv_heads, PAGE, self.head_dim)),
                PagedTensor("v", (self.num_kv_heads, self.head_dim, PAGE)))


@dataclass(frozen=True)
class StateSpec:
    """State of fixed size per request (shape without the slot dimension)."""

    shape: tuple
    dtype: torch.dtype = torch.float32


# --------------------------------------------------------------------------- step context
@dataclass
class StepContext:
    """What one step's kernels need to know about the batch; built by the step function.

    Device tensors are int32.  ``T`` tokens belong to ``R`` requests; request r owns
    tokens ``q_start[r] .. q_start[r+1]``, at absolute positions
    ``kv_len[r] - q_len[r] ..  kv_len[r] - 1``.
    """

    T: int
    R: int
    dtype: torch.dtype                    # compute / activation dtype
    token_ids: torch.Tensor               # [T]
    positions: torch.Tensor               # [T] absolute position of each token
    req_of_token: torch.Tensor            # [T] row of the token's request in this step
    q_start: torch.Tensor                 # [R+1]
    kv_len: torch.Tensor                  # [R] keys visible after this step's writes
    slots: torch.Tensor                   # [R] per-request state slot
    block_tables: Dict[int, torch.Tensor]  # cache group -> [R, width] page ids (-1 = none)
    logit_rows: torch.Tensor              # [M] token rows whose logits are wanted
    uneven: Optional[torch.Tensor] = None  # [1] 1: the requests' lengths are uneven (ops.lengths_uneven); None: nobody says
    # host-side copies for launch planning (never read by kernels)
    q_lens: Sequence[int] = ()
    kv_lens: Sequence[int] = ()
    max_q_len: int = 0
    max_kv_len: int = 0
    all_decode: bool = False
    every_row: bool = False               # a step of single tokens whose logits are all wanted: logit_rows are 0 .. T - 1
    host_slots: Sequence[int] = ()        # the requests' state slots, on the host
    # Set by whoever arranges the parts, for the part that runs next: it may leave its update of
    # the stream in pieces (``ops.gemm(..., may_defer=True)``) because the stream's next reader
    # adds them.  False unless an arrangement says so, so a part never defers by itself.
    may_defer: bool = False
    # Set beside ``may_defer``, or None: (weight, eps) of the norm that reads the stream next, when that norm's own reader takes
    # a norm whose root is left to it (``ops.gemm(..., next_norm=...)``).
    next_norm: Any = None
    opening_norm: Any = None              # set by the model for the embedding: (weight, eps, dtype) of the norm that reads the stream first
    after_block_norm: Any = None          # set by the model per block: ``next_norm`` for whoever reads the stream after this block
    may_leave_choices: bool = False       # likewise: a routed feed-forward may leave its result as the experts' rows (``ops.LeftChoices``)
    after_block_consumes: bool = False    # set by the model per block: whoever reads the stream after this block adds pending pieces
    read_rows: Optional[torch.Tensor] = None  # set for a mixer that ``cuts_rows``: the only rows of the stream that are read after it
    workspace: Any = None                 # the runner's ops.KernelWorkspace: scratch memory of the kernels
    plans: Dict[Any, Any] = field(default_factory=dict)     # step planner -> what it made for this step
    scratch: Dict[Any, Any] = field(default_factory=dict)   # what parts share within one step; emptied per step


@dataclass
class LayerCache:
    """The view of the cache manager that one entry of the run order gets."""

    group: int = -1                       # cache group of the pages (-1: no pages)
    k: Optional[torch.Tensor] = None      # [pages, kv_heads, page_size, head_dim]   (= tensors["k"])
    v: Optional[torch.Tensor] = None      # [pages, kv_heads, head_dim, page_size]   (= tensors["v"])
    page_size: int = 0
    writes: bool = True                   # False: reads another entry's cache
    state: Optional[torch.Tensor] = None  # [max_slots, *StateSpec.shape]
    tensors: Dict[str, torch.Tensor] = field(default_factory=dict)   # every paged tensor by name: [pages, *page shape]


def says_of_rows(part: Any, name: str) -> bool:
    """What ``part``'s class says of rows that nobody reads, unless the object's ``forward`` has been replaced by another."""
    return "forward" not in vars(part) and bool(getattr(part, name, False))


def cut_rows(ctx: StepContext, *tensors: torch.Tensor):
    """Copies of the rows of ``tensors`` that ``ctx.read_rows`` names (what has only them already, from a mixer beside, as it is:
    they are half of the step's tokens at most)."""
    rows = ctx.read_rows
    made = iter(ops.copy_rows(rows, *(t for t in tensors if t.shape[0] != rows.shape[0])))
    return tuple(t if t.shape[0] == rows.shape[0] else next(made) for t in tensors)


# --------------------------------------------------------------------------- part bases
class Part:
    """Common behaviour: declare tensors, receive them, know the compute dtype.

    ``graph_safe``: True promises that ``forward`` does the same launches, on the same addresses,
    for every step of one batch size of single tokens - it reads nothing of the step on the host
    (``ctx.host_slots``, ``ctx.q_lens``, ``ctx.kv_lens``, values of device tensors) and decides
    nothing in Python from it.  Only then may a decode step be captured once as a HIP graph and
    replayed; one part without the promise makes the whole model step eagerly.  The default is
    False: a part has to say so.

    What a class says of norms that are left to their reader (``leaves_root``, ``takes_left_norm``; a block's ``first_norm``
    and ``opening_norm``) and of rows that nobody reads (``rowwise``, ``cuts_rows``, ``ends_in_rows``) it says of its own
    ``forward``: a subclass with another ``forward`` says it again or does not.
    """

    graph_safe = False

    def __init_subclass__(cls, **kwargs):
        super().__init_subclass__(**kwargs)
        if "forward" in cls.__dict__:
            for name, nothing in (("leaves_root", False), ("takes_left_norm", False), ("first_norm", None), ("opening_norm", None),
                                  ("rowwise", False), ("cuts_rows", False), ("ends_in_rows", False)):
                if name not in cls.__dict__:
                    setattr(cls, name, nothing)

    def tensor_specs(self) -> List[TensorSpec]:
        return []

    def load(self, tensors: Dict[str, torch.Tensor], dtype: torch.dtype, device: torch.device) -> None:
        """Receive this part's tensors (relative names), already on ``device``."""
        self.dtype = dtype
        self.device = device

    def streamed_weights(self) -> List[torch.Tensor]:
        """After ``load``: the weight matrices [out, in] that this part hands to ``ops.gemm`` /
        ``ops.gemm_swiglu`` whole, in every decode step.  Whoever runs the model may keep a second
        copy of each in the order the weight-streaming kernels read (``EngineOptions.stream_copies``);
        a part that names none loses nothing but that."""
        return []

    def norm_readers(self) -> List[torch.Tensor]:
        """Of a part that takes left norms: the matrices that multiply its activations.  A norm is left to it only where every
        one of these products applies the root, which those with a streaming copy do."""
        return self.streamed_weights()


class Norm(Part):
    leaves_root = False        # True: ``forward`` returns an ``ops.LeftNorm`` where the product before it has left one

    def forward(self, x: torch.Tensor, ctx: Optional[StepContext] = None, rows: Optional[torch.Tensor] = None) -> torch.Tensor:
        """``x`` float32 [N, D] -> normalised rows in the compute dtype ([M, D] when
        ``rows`` (int32 [M]) selects rows of ``x``).  ``ctx`` is the step's context (None
        when the norm is used on its own)."""
        raise NotImplementedError


class PositionEncoding(Part):
    """Encodes positions into queries and keys.

    ``rotary_params()`` lets the attention mixer fuse the rotation into its cache-write
    kernel; a scheme that is not a rotation returns None and implements ``apply``.
    """

    def rotary_params(self, ctx=None):
        return None

    def apply(self, q: torch.Tensor, k: torch.Tensor, ctx: StepContext) -> None:
        raise NotImplementedError


class Mixer(Part):
    takes_left_norm = False    # True: ``forward`` takes an ``ops.LeftNorm`` for its activations (its products of them do)
    cuts_rows = False          # True: where ``ctx.read_rows`` names rows, ``forward`` updates a copy of them alone and returns it

    def cache_spec(self):
        """What the mixer keeps per request: ``KVCacheSpec`` / ``PagedCacheSpec`` (per token, in
        pages), ``StateSpec`` (fixed size), or None."""
        return None

    def step_planner(self, page_size: int):
        """Called once after ``load``.  A mixer whose kernels want host-made work lists per step
        returns a hashable *planner* with ``plan(q_lens, kv_lens) -> None | (arrays, finish)``:
        ``arrays`` are int32 numpy arrays by name, which the step function packs into its one
        upload of metadata, and ``finish(views)`` turns their device views into whatever the
        mixer reads back from ``ctx.plans[planner]``.  Planners that compare equal run once per
        step, for all their mixers.  None: nothing to plan."""
        return None

    def forward(self, h: torch.Tensor, x: torch.Tensor, ctx: StepContext, cache: LayerCache) -> Optional[torch.Tensor]:
        """Read activations ``h`` [T, D]; add the mixer's output into ``x`` (float32).  A mixer that ``cuts_rows`` returns what
        it has added to: ``x``, or where ``ctx.read_rows`` was set those rows alone, of which ``x`` may hold no others."""
        raise NotImplementedError


class FeedForward(Part):
    takes_left_norm = False    # as a mixer's
    rowwise = False            # True: a token's result takes nothing from other tokens, nor from what ``ctx`` says of them

    def forward(self, h: torch.Tensor, x: torch.Tensor, ctx: StepContext) -> None:
        """Read activations ``h`` [T, D]; add the result into ``x`` (float32)."""
        raise NotImplementedError


class Block(Part):
    """An arrangement of norm(s), mixer(s) and feed-forward around the residual stream.

    The stream a block receives is finished (no update pending) unless the block says that its
    first reader adds pending pieces (``reads_deferred``), and no part inside it leaves an update
    pending unless the block sets ``ctx.may_defer`` before calling it.  An arrangement that knows
    nothing of deferred updates therefore never meets one."""

    mixer: Mixer
    takes_left_join = False    # True: the block's first reader applies a result that a sandwich block has left (``norm.LEFT_JOIN``)
    reads_deferred = False     # True: the block's first reader of the stream is a norm that adds pending pieces
    ends_in_rows = False       # True: the block has a ``forward_last(x, ctx, cache)``: as ``forward``, the stream after it only at ``ctx.logit_rows``

    @property
    def first_norm(self):
        """(the norm that reads the stream first, the part that reads the norm), where the one may be left to the other; else None."""
        return None

    def mixers(self) -> List[Mixer]:
        """The block's mixers - and other parts of it that keep something per request (they have a mixer's
        ``cache_spec`` and ``step_planner``) - each with a cache or state of its own.  With more than one, ``forward``
        receives a list of ``LayerCache`` in this order instead of a single one."""
        m = getattr(self, "mixer", None)
        return [m] if m is not None else []

    @property
    def opening_norm(self):
        """(weight, eps, dtype) of the RMS norm that reads the stream first, when whoever makes the stream may make it too; else None."""
        return None

    def forward(self, x: torch.Tensor, ctx: StepContext, cache) -> None:
        raise NotImplementedError


# --------------------------------------------------------------------------- registries
class PartRegistry:
    def __init__(self, what: str):
        self.what = what
        self._makers: Dict[str, Callable[..., Any]] = {}

    def register(self, kind: str, maker: Callable[..., Any] | None = None):
        """``register("name", cls)`` or ``@register("name")``."""
        if maker is None:
            def deco(m):
                self._makers[kind] = m
                return m
            return deco
        self._makers[kind] = maker
        return maker

    def make(self, kind: str, **params) -> Any:
        if kind not in self._makers:
            known = ", ".join(sorted(self._makers)) or "<none>"
            raise UnsupportedModelError(f"{self.what} '{kind}' is not registered (registered: {known})")
        return self._makers[kind](**params)

    def kinds(self) -> tuple:
        return tuple(sorted(self._makers))


NORMS = PartRegistry("norm")
MIXERS = PartRegistry("mixer")
FEED_FORWARDS = PartRegistry("feed-forward")
POSITION_ENCODINGS = PartRegistry("position encoding")
BLOCKS = PartRegistry("block arrangement")
