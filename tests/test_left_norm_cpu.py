"""Norms whose root is left to their reader: when what was left still counts (CPU)."""
import pytest
import torch

from photon_infer_amd import ops
from photon_infer_amd.errors import KernelError
from photon_infer_amd.ops.workspace import LeftNorm

F32, BF16 = torch.float32, torch.bfloat16


def left_in(ws, x, weight):
    ws.left_norm = LeftNorm(x, weight, 1e-5, (x * weight).to(BF16), (x ** 2).sum(1, keepdim=True), 1)
    return ws.left_norm


def test_a_stream_that_somebody_wrote_has_no_norm_left():
    ws, weight = ops.KernelWorkspace("cpu"), torch.ones(8)
    for write in (lambda x: x.add_(1), lambda x: x[1].mul_(2), lambda x: x.view(-1)[:3].zero_(), lambda x: x.copy_(torch.ones(2, 8)), ops._changes):
        x = torch.randn(2, 8)
        left = left_in(ws, x, weight)
        assert ws.take_left_norm(x, weight, 1e-5) is left and ws.left_norm is None
        left = left_in(ws, x, weight)
        write(x)
        assert ws.take_left_norm(x, weight, 1e-5) is None and ws.left_norm is None
        with pytest.raises(KernelError, match="written since"):
            ops.whole_norm(left)


def test_tensors_that_count_no_versions_keep_their_norms():
    with torch.inference_mode():
        ws, weight, x = ops.KernelWorkspace("cpu"), torch.ones(8), torch.randn(2, 8)
        left = left_in(ws, x, weight)
        ops._changes(x)                                  # not an error
        assert ws.take_left_norm(x, weight, 1e-5) is left


def test_a_subclass_with_another_forward_makes_no_promise_by_inheritance():
    """A norm, feed-forward or arrangement that wraps one of the framework's own works on tensors and finished streams,
    as it does beside parts that leave nothing."""
    from photon_infer_amd.parts.block import PreNormBlock
    from photon_infer_amd.parts.mlp import SwiGLU
    from photon_infer_amd.parts.norm import RMSNorm, norm_left_to

    class DoubledNorm(RMSNorm):
        def forward(self, x, ctx=None, rows=None):
            return super().forward(x, ctx, rows) * 2

    class RoundedMLP(SwiGLU):
        def forward(self, h, x, ctx):
            super().forward(h.round(), x, ctx)

    class Same(RMSNorm):
        pass

    class ShiftedBlock(PreNormBlock):
        def forward(self, x, ctx, cache):
            super().forward(x.add_(2), ctx, cache)

    class Says(RoundedMLP):
        takes_left_norm = True

        def forward(self, h, x, ctx):
            SwiGLU.forward(self, h, x, ctx)

    def norm(kind):
        n = kind(8, 1e-5)
        n.load({"weight": torch.ones(8, dtype=BF16)}, BF16, torch.device("cpu"))
        return n

    def mlp(kind):
        m = kind(64, 16)
        m.w_gate_up = torch.zeros(32, 64, dtype=BF16)
        assert ws.add_stream_copy(m.w_gate_up)
        return m

    ws = ops.KernelWorkspace("cpu")
    assert norm_left_to(norm(RMSNorm), mlp(SwiGLU), ws) is not None and norm_left_to(norm(Same), mlp(SwiGLU), ws) is not None
    assert norm_left_to(norm(DoubledNorm), mlp(SwiGLU), ws) is None and norm_left_to(norm(RMSNorm), mlp(RoundedMLP), ws) is None
    assert norm_left_to(norm(RMSNorm), mlp(Says), ws) is not None
    for kind, leaves in ((PreNormBlock, True), (ShiftedBlock, False)):
        block = kind(("n.", norm(RMSNorm)), ("m.", SwiGLU(64, 16)))
        assert (block.first_norm is not None) == leaves and (block.opening_norm is not None) == leaves, kind


def test_a_sum_does_not_take_a_left_norm():
    """Refused before anything is launched: no kernel is compiled for it (``ops.gemm`` makes the whole norm there)."""
    from photon_infer_amd.ops import _lib, fast
    A = 1 << 20                                          # addresses that nobody reads
    with pytest.raises(KernelError, match="does not take a left norm"):
        _lib.call("bf16", "pi_gemm_rows", A, fast.EPI_ACCUM, 64, A, 64, A, 1, 64, 64, A, 8, 1e-5, None)


def test_a_norm_is_left_only_where_every_product_of_it_applies_the_root():
    from photon_infer_amd.parts.block import SideBySide
    from photon_infer_amd.parts.delta_rule import ChannelDeltaRule
    from photon_infer_amd.parts.embedding import LMHead
    from photon_infer_amd.parts.mlp import ClampedGLU, SwiGLU
    from photon_infer_amd.parts.norm import RMSNorm, norm_left_to
    n = RMSNorm(64, 1e-5)
    n.load({"weight": torch.ones(64, dtype=BF16)}, BF16, torch.device("cpu"))
    mat = lambda rows: torch.zeros(rows, 64, dtype=BF16)

    def delta(rows, low):
        d = ChannelDeltaRule(64, 4, 4, 16, 16, 4, 16, 16, 1e-5)
        d.w_in, d.w_low = mat(rows), mat(low)
        return d

    def with_matrix(part, name, rows):
        setattr(part, name, mat(rows))
        return part

    for make, fits in ((lambda: with_matrix(SwiGLU(64, 16), "w_gate_up", 32), True), (lambda: with_matrix(ClampedGLU(64, 16, 7.0), "w_gate_up", 32), True),
                       (lambda: with_matrix(SwiGLU(64, 20), "w_gate_up", 40), False), (lambda: with_matrix(LMHead(32, 64, False), "weight", 32), True),
                       (lambda: with_matrix(LMHead(33, 64, False), "weight", 33), False), (lambda: delta(208, 32), True), (lambda: delta(196, 32), False),
                       (lambda: delta(208, 40), False), (lambda: SideBySide([("a.", delta(208, 32)), ("b.", delta(208, 32))]), True),
                       (lambda: SideBySide([("a.", delta(208, 32)), ("b.", delta(196, 32))]), False)):
        part = make()
        for copies in (False, True):
            ws = ops.KernelWorkspace("cpu")
            for w in part.norm_readers() if copies else []:
                ws.add_stream_copy(w)
            assert (norm_left_to(n, part, ws) is not None) == (fits and copies), (type(part).__name__, copies)
        assert norm_left_to(n, part, None) is None


def test_a_subclass_with_another_forward_says_nothing_of_rows_by_inheritance():
    """Whoever mixes tokens in a feed-forward, mixer or arrangement of its own gets all of them."""
    from photon_infer_amd.parts.attention import PagedAttention
    from photon_infer_amd.parts.block import PreNormBlock
    from photon_infer_amd.parts.mlp import GeluMLP, SwiGLU

    class Mixes(SwiGLU):
        def forward(self, h, x, ctx):
            super().forward(h + h.roll(1, 0), x, ctx)

    class Named(SwiGLU):
        pass

    class Averaged(PagedAttention):
        def forward(self, h, x, ctx, cache):
            super().forward(h, x, ctx, cache)
            x.sub_(x.mean(0))

    class Scaled(PreNormBlock):
        def forward(self, x, ctx, cache):
            super().forward(x, ctx, cache)
            x.mul_(2)

    assert SwiGLU.rowwise and Named.rowwise and GeluMLP.rowwise and not Mixes.rowwise
    assert not Averaged.cuts_rows and not Scaled.ends_in_rows
    from photon_infer_amd.parts.base import says_of_rows
    wrapped = SwiGLU(8, 16)
    assert says_of_rows(wrapped, "rowwise")
    wrapped.forward = lambda h, x, ctx: None
    assert not says_of_rows(wrapped, "rowwise")
